// One compute step of the quantized ring all-reduce on one chunk of the bucket, for gfx950.
//
// The ring schedule of the reference (ccdl_comm/cuda/transports/pipelined_ring.py:216-275) alternates, on every
// rank, "decode the payload that arrived into chunk c of the bucket" with "quantize chunk c and send it on":
// the chunk a step reduces into is always the chunk the next step sends.  The reference runs these as two
// kernels (ccdl_comm/cuda/transports/torch_topology.py:236-316: dequantize with reduce_op sum or none, an in-place
// division at the last reduce step, then quantize), which reads the chunk twice and writes it once.  Here the
// updated chunk is quantized while it is still in registers: one launch reads the received payload and the
// chunk, writes the chunk and the next payload.
//
// Per element, in the order the two-kernel sequence rounds:
//   d = T(float(code) * scale)                  decode, rounded to the chunk's type T
//   v = T(float(chunk) + d)      (ACC only)     the in-place sum in T arithmetic
//   v = T(v / divisor)           (divisor != 1) the in-place mean (divide_all)
//   chunk = v;  payload = quantize(v)           same group maximum, scale and rounding as quant_pack_kernel
//
// A hop that does not complete the sum has no use for the updated chunk beyond its payload: the ring's second phase
// overwrites the chunk before anything reads it.  Without the write-back (keep = 0) such a hop moves a third fewer bytes;
// GPU time of a ring of eight ranks, fourteen hops: 13.1 M bf16 elements 48.4 -> 47.4 us, 26.2 M 65.1 -> 60.4, 6.6 M fp32
// 43.4 -> 42.0.
//
// Mapping: one lane owns 16 bytes of the chunk (4 fp32 or 8 16-bit elements), a group sits in adjacent lanes of
// one DPP row, a 256-thread block walks UNROLL * 4 wavefront tiles with every load issued before the first use.
#include <type_traits>

#include "device_utils.h"
#include "launch.h"

namespace lbc {
namespace {

// Tiles in flight per wavefront beyond the chip's wavefront slots: one, except for the write-only step on a 16-bit chunk,
// which keeps two (decode only, 26.2 M bf16 elements 13.6 us with two, 14.2 with one; decode + requantize 15.8 / 16.1).
// An fp32 chunk's write-only step used to keep four: 26.2 M elements 23.5 us, with one 22.3; 6.6 M 7.8 and 7.0 us.
template <typename T, bool ACC> constexpr int ring_unroll() { return ACC || sizeof(T) == 4 ? 1 : 2; }
template <typename T, int TILES> struct ring_tiling {
    static constexpr int VEC = 16 / sizeof(T);
    static constexpr int TILE = kWave * VEC;
    static constexpr int UNROLL = TILES;
    static constexpr int BLOCK_ELEMS = TILE * kWavesPerBlock * UNROLL;
};

template <typename T, int G, int MODE, bool ACC, int TILES>
__global__ __launch_bounds__(kBlock) void ring_step_kernel(const RingStepArgs a) {
    using L = ring_tiling<T, TILES>;
    constexpr int VEC = L::VEC;
    constexpr int LPG = G / VEC;
    constexpr int UNROLL = L::UNROLL;
    static_assert(LPG >= 1 && LPG <= 16, "a group must fit one DPP row");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t padded = (a.numel + G - 1) / G * G;
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(L::BLOCK_ELEMS)) * L::BLOCK_ELEMS;
    if (block_first >= padded) return;

    T *chunk = static_cast<T *>(a.chunk);  // read and written by the same lane: no restrict
    const int8_t *__restrict__ recv_codes = a.recv_codes;
    const float *__restrict__ recv_scales = a.recv_scales;
    const bool mean = a.divisor != 1.0f;
    const bool emit = a.send_codes != nullptr, keep = a.keep != 0;  // uniform over the grid

    // WHOLE: all of the block's elements exist; otherwise a lane's vector is cut short at the end of the chunk, and
    // what lies behind it counts as zeros (every lane of a row takes part in the group maximum).  The element-wise walk
    // this replaces bounded every chunk that is no whole number of blocks and every chunk off a 16-byte line: 822,623
    // bf16 elements, decode + requantize, 5.7 us then, 3.1 us now; 6,553,601 fp32 elements at an odd start 21.8 and
    // 9.0 us (9.5 us without the non-temporal hint on the stores), with the sum 26.0 and 12.7 us.
    auto tiles = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        // Whole blocks of aligned chunks use one descriptor per stream over the block's span and 32-bit offsets per lane: GPU time of
        // the ring of eight ranks on 13.1 M bf16 elements 46.6 -> 46.2 us, 26.2 M 59.0 -> 58.6, 6.6 M fp32 41.5 -> 41.3.  (Written
        // through beside the hint, the chunk's stores are 0.3 us faster on 13.1 M and 0.4 slower on the others; the codes' 1 to 2 us slower.)
        constexpr bool BUFFERS = WHOLE && MODE != kUnaligned;
        constexpr bool kNt = MODE == kStream || MODE == kUnaligned;
        constexpr int kPolicy = policy_of<MODE>();
        constexpr int kCodeAlign = MODE == kUnaligned ? 1 : VEC;
        const buffer_t recv_codes_b = buffer_over(recv_codes + block_first, L::BLOCK_ELEMS);
        const buffer_t recv_scales_b = buffer_over(recv_scales + block_first / G, L::BLOCK_ELEMS / G * 4);
        const buffer_t chunk_b = buffer_over(chunk + block_first, L::BLOCK_ELEMS * sizeof(T));
        T xv[UNROLL][VEC];
        uint32_t words[UNROLL][VEC / 4];
        float rscale[UNROLL];
        int64_t e0[UNROLL];
        uint32_t at[UNROLL];   // element offset inside the block
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            at[u] = static_cast<uint32_t>(tile_in_block<UNROLL>(u, wave)) * L::TILE + lane * VEC;
            e0[u] = block_first + at[u];
#pragma unroll
            for (int k = 0; k < VEC / 4; ++k) words[u][k] = 0;
            rscale[u] = 0.0f;
            // The one code stream is a fifth of the traffic at most; without the non-temporal hint it measures
            // faster, as in the single-payload decode kernel.
            if constexpr (BUFFERS) {
                buffer_load<uint32_t, VEC / 4, kCached>(recv_codes_b, at[u], words[u]);
                float one[1];
                buffer_load<float, 1, kCached>(recv_scales_b, at[u] / G * 4, one);
                rscale[u] = one[0];
            } else if (WHOLE || e0[u] < a.numel) {
                load_any<uint32_t, VEC / 4, false, kCodeAlign>(reinterpret_cast<const uint32_t *>(recv_codes + e0[u]), words[u]);
                rscale[u] = recv_scales[e0[u] / G];
            }
            if constexpr (ACC && BUFFERS) buffer_load<T, VEC, kPolicy>(chunk_b, at[u] * sizeof(T), xv[u]);
            else if constexpr (ACC && WHOLE) load_any<T, VEC, kNt>(chunk + e0[u], xv[u]);
            else if constexpr (ACC) load_live<T, VEC, kNt>(chunk + e0[u], a.numel - e0[u], xv[u]);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            float p[VEC];
            T out[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) p[i] = code_to_float(words[u][i / 4], i % 4) * rscale[u];
            round_through_all<T, VEC>(p);
            if constexpr (ACC) {
#pragma unroll
                for (int i = 0; i < VEC; ++i) p[i] = widen(xv[u][i]) + p[i];
                round_through_all<T, VEC>(p);
            }
            if (mean) divide_all<T, VEC>(p, a.divisor);
            narrow_all<T, VEC>(p, out);
            if constexpr (WHOLE) {
                if (!ACC || keep) {
                    if constexpr (BUFFERS) buffer_store<T, VEC, kPolicy>(chunk_b, at[u] * sizeof(T), out);
                    else store_any<T, VEC, kNt>(chunk + e0[u], out);
                }
            } else {
                if (!ACC || keep) store_live<T, VEC, kNt>(chunk + e0[u], a.numel - e0[u], out);
#pragma unroll
                for (int i = 0; i < VEC; ++i) p[i] = e0[u] + i < a.numel ? p[i] : 0.0f;
            }
            if (emit) {
                const float scale = group_scale<VEC, LPG>(p);
                int c[VEC];
                encode_group<VEC>(p, scale, c);
                uint32_t packed[VEC / 4];
#pragma unroll
                for (int k = 0; k < VEC / 4; ++k) packed[k] = pack4(c[4 * k], c[4 * k + 1], c[4 * k + 2], c[4 * k + 3]);
                if constexpr (BUFFERS) {
                    buffer_store<uint32_t, VEC / 4, kPolicy>(buffer_over(a.send_codes + block_first, L::BLOCK_ELEMS), at[u], packed);
                    const float one[1] = {scale};
                    if ((lane & (LPG - 1)) == 0) buffer_store<float, 1, kCached>(buffer_over(a.send_scales + block_first / G, L::BLOCK_ELEMS / G * 4), at[u] / G * 4, one);
                } else if (WHOLE || e0[u] < padded) {
                    store_any<uint32_t, VEC / 4, kNt, kCodeAlign>(reinterpret_cast<uint32_t *>(a.send_codes + e0[u]), packed);
                    if ((lane & (LPG - 1)) == 0) a.send_scales[e0[u] / G] = scale;
                }
            }
        }
    };
    if (block_first + L::BLOCK_ELEMS <= a.numel) tiles(std::true_type{});
    else tiles(std::false_type{});
}

template <typename T, int G, bool ACC, int TILES>
hipError_t launch_ring_tiles(int mode, const RingStepArgs &a, hipStream_t stream) {
    using L = ring_tiling<T, TILES>;
    const int64_t padded = (a.numel + G - 1) / G * G;
    const int64_t blocks = (padded + L::BLOCK_ELEMS - 1) / L::BLOCK_ELEMS;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    switch (mode) {
        case kStream: hipLaunchKernelGGL((ring_step_kernel<T, G, kStream, ACC, TILES>), grid, dim3(kBlock), 0, stream, a); break;
        case kVector: hipLaunchKernelGGL((ring_step_kernel<T, G, kVector, ACC, TILES>), grid, dim3(kBlock), 0, stream, a); break;
        default: hipLaunchKernelGGL((ring_step_kernel<T, G, kUnaligned, ACC, TILES>), grid, dim3(kBlock), 0, stream, a); break;
    }
    return hipGetLastError();
}

// One tile a wavefront while the tiles fit the chip's wavefront slots (decode + requantize, us with one / two tiles: 65,536
// bf16 elements 2.0 / 2.3, 1 Mi 2.7 / 3.0, 4 Mi 4.1 / 4.3, 6.6 M 5.4 / 5.4).
template <typename T, int G, bool ACC>
hipError_t launch_ring_g(int mode, const RingStepArgs &a, hipStream_t stream) {
    constexpr int TILES = ring_unroll<T, ACC>();
    if (TILES > 1 && a.numel <= kResidentWaves * ring_tiling<T, 1>::TILE) return launch_ring_tiles<T, G, ACC, 1>(mode, a, stream);
    return launch_ring_tiles<T, G, ACC, TILES>(mode, a, stream);
}

template <typename T>
hipError_t launch_ring_t(int g, bool accumulate, int mode, const RingStepArgs &a, hipStream_t s) {
    switch (g) {
        case 64: return accumulate ? launch_ring_g<T, 64, true>(mode, a, s) : launch_ring_g<T, 64, false>(mode, a, s);
        case 32: return accumulate ? launch_ring_g<T, 32, true>(mode, a, s) : launch_ring_g<T, 32, false>(mode, a, s);
        case 16: return accumulate ? launch_ring_g<T, 16, true>(mode, a, s) : launch_ring_g<T, 16, false>(mode, a, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace

hipError_t launch_ring_step(int dtype, int group_size, bool accumulate, int mode, const RingStepArgs &args,
                            hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_ring_t<float>(group_size, accumulate, mode, args, stream);
        case kF16: return launch_ring_t<f16>(group_size, accumulate, mode, args, stream);
        case kBF16: return launch_ring_t<bf16>(group_size, accumulate, mode, args, stream);
        default: return hipErrorNotSupported;
    }
}

}  // namespace lbc
