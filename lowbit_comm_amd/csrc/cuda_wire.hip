// Kernels for the payload format of the reference's CUDA extension (ccdl_cuda_ops), so that
// gfx950 ranks can exchange payloads with ranks running that extension.
//
// Format (ccdl_comm/csrc/quantization/quant_pack_kernel.cu:101-162 writes it,
// dequant_reduce_kernel.cu:27-69 reads it), for element type T of the tensor:
//   scale of a group  = max |p| over the group, stored as T (NaNs skipped, fmaxf);
//   code              = rint(p * (127 / max(float(scale), 1e-6f))), NaN -> 0;
//   bytes of a group  = codes with the byte order reversed inside every sizeof(T)-byte word
//                       (2-byte words for fp16/bf16, 4-byte words for fp32);
//   compact layout    = per group [G code bytes][scale]; otherwise all code bytes, then all scales;
//   decode            = float(code) * (float(scale) / 127), rounded to T.
// 4-bit codes (BIT = 4; quant_pack_kernel.cu:103,120-130,145-158, inner.cuh:36-40): multiplier
// 7 / max(scale, 1e-6), two's-complement nibbles, 2*sizeof(T) codes per word with the first code in
// the most significant nibble, decode by scale / 7; quantize and single-payload decode only, as in
// the reference (its fused reduce is 8-bit).
//
// Mapping: as in the portable-format kernels, one lane owns 16 bytes of the tensor (4 fp32 or
// 8 half elements), a group sits in adjacent lanes of one DPP row, and every tile's loads are
// issued before the arithmetic.  Group strides of 66 or 68 bytes leave code words only 2- or
// 4-byte aligned; gfx950 global memory instructions accept that, so all accesses here are typed
// with element alignment only and there is no separate path for unaligned tensors.
#include <type_traits>

#include "device_utils.h"
#include "launch.h"
#include "wire_common.h"

// Chunk size (log2 of the element count) from which the gather hop of interleaved 16-bit payloads stores group pairs
// as shifted dwords; below it the misaligned 8-byte stores measured faster (see wire_ring_step_kernel).
#ifndef LBC_PAIR_STORE_MIN_LOG2
#define LBC_PAIR_STORE_MIN_LOG2 22
#endif


namespace lbc {
namespace {

// ---------------------------------------------------------------------------
// quantize + pack (optionally x + residual), `world` chunks via blockIdx.y
// ---------------------------------------------------------------------------
// Code stores beside kPlain and kNonTemporal: written through the L2 (fp32 tensors, 8-bit codes apart from the scales).
constexpr int kWrittenThrough = 2;

// NT: hint of the tensors' loads; CODES: how the codes leave (launch_wire_quant_c).  The sum is read again by the reduce that
// follows: plain stores, 6.6 M elements of two payloads through the all_gather hook with error feedback 31.4 -> 29.0 us (fp32)
// and 19.9 -> 17.3 (bf16), 20 M of eight 109 -> 104 and 75.7 -> 73.0; interleaved 16-bit payloads, which gain nothing,
// keep the hint (6.6 M of four 22.8 against 23.2 us).
template <typename T, int G, int BIT, bool HAS_R, bool COMPACT, int NT, int CODES, int TILES>
__global__ __launch_bounds__(kBlock) void wire_quant_kernel(const WireQuantArgs a) {
    constexpr int SUM_NT = COMPACT && sizeof(T) == 2 ? NT : kPlain;
    using W = wire<T, BIT>;
    constexpr int VEC = W::VEC;
    constexpr int LPG = G / VEC;
    constexpr int UNROLL = TILES;
    constexpr int BLOCK_ELEMS = W::TILE * kWavesPerBlock * UNROLL;
    static_assert(LPG >= 1 && LPG <= 16, "a group must fit one DPP row");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t chunk = blockIdx.y;
    const int64_t chunk_start = chunk * a.shard_numel;
    int64_t valid = a.numel - chunk_start;
    valid = valid < 0 ? 0 : (valid > a.shard_numel ? a.shard_numel : valid);
    const int64_t groups = (a.shard_numel + G - 1) / G;
    const int64_t padded = groups * G;
    const group_layout<T, G, COMPACT, BIT> at{groups};
    // The reference sends a chunk of whole groups without a residual to its general kernels, whose running
    // maximum a NaN resets, and everything else to the fused pack kernel, whose fmaxf skips NaNs
    // (quant_pack_kernel.cu:231,259-262).
    // With `prepared` the call stands for torch's add, zero padding to whole groups and a quantize without residual.
    // Bound by memory, 13 bytes an element of fp32 where the two calls move 17: the all_gather hook with error feedback on
    // 6.6 M fp32 elements and eight payloads 43.3 us with two calls, 39.3 us with one.
    T *prepared = HAS_R ? static_cast<T *>(a.prepared) : nullptr;
    const bool resets = a.nan_resets != 0 && (prepared != nullptr || (!HAS_R && valid % G == 0));

    const T *__restrict__ x = static_cast<const T *>(a.x) + chunk_start;
    const T *__restrict__ r = HAS_R ? static_cast<const T *>(a.residual) + chunk_start : nullptr;
    uint8_t *__restrict__ payload = a.payloads + chunk * a.payload_stride;

    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(BLOCK_ELEMS)) * BLOCK_ELEMS;
    if (block_first >= padded) return;

    using Raw = typename raw_bits<T>::type;
    auto multiplier_of = [&](float absmax) {
        const float scale = absmax < 1.0e-6f ? 1.0e-6f : absmax;   // a NaN stays and zeroes every code
        return W::LEVELS / scale;
    };
    auto group_multiplier = [&](uint32_t absmax_bits, float &absmax) {
        absmax = as_f32(group_max_bits<LPG>(absmax_bits));
        return multiplier_of(absmax);
    };
    // The scale of the lane's group as the reference's general kernels compute it, from the elements as stored.
    auto scan_scale = [&](const T (&elements)[VEC], int64_t group, int k0) {
        uint32_t mag[VEC];
#pragma unroll
        for (int i = 0; i < VEC; ++i) mag[i] = __builtin_bit_cast(Raw, elements[i]) & raw_bits<T>::ABS;
        return running_max_raw<T, G, VEC>(mag, k0, scan_start<T, G>(group));
    };
    auto clamp_codes = [&](int (&c)[VEC]) {
        constexpr int L = static_cast<int>(W::LEVELS);
#pragma unroll
        for (int i = 0; i < VEC; ++i) c[i] = c[i] < -L ? -L : (c[i] > L ? L : c[i]);
    };

    // One pass over the block's tiles, every load issued before the first use.  WHOLE: all of the block's elements are
    // live; otherwise a lane's vector is cut short where the chunk ends, and what lies behind counts as zeros
    // (walked element by element, the last block bounded every small tensor: 10,048 bf16 elements 2.5 us, now 2.0 us).
    auto tiles = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        T xv[UNROLL][VEC];
        T rv[UNROLL][VEC];
        int64_t e0[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            e0[u] = block_first + static_cast<int64_t>(tile_in_block<UNROLL>(u, wave)) * W::TILE + lane * VEC;
            if constexpr (WHOLE) {
                load_elems<T, VEC, NT>(x + e0[u], xv[u]);
                if constexpr (HAS_R) load_elems<T, VEC, NT>(r + e0[u], rv[u]);
            } else {
                load_live<T, VEC, NT == kNonTemporal>(x + e0[u], valid - e0[u], xv[u]);
                if constexpr (HAS_R) load_live<T, VEC, NT == kNonTemporal>(r + e0[u], valid - e0[u], rv[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            float p[VEC];
            uint32_t m = 0;   // largest magnitude pattern; above the pattern of infinity when the lane holds a NaN
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                p[i] = widen(xv[u][i]);
                if constexpr (HAS_R) p[i] += widen(rv[u][i]);
            }
            if constexpr (HAS_R) round_through_all<T, VEC>(p);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const uint32_t bits = as_u32(p[i]) & 0x7FFFFFFFu;
                m = bits > m ? bits : m;
            }
            const bool nans = __ballot(m > 0x7F800000u) != 0;   // somewhere in the wavefront: rare, and uniform
            T held[VEC];   // the elements as stored
            if constexpr (HAS_R) {
                narrow_all<T, VEC>(p, held);
                if (same_t<T, bf16>::value && nans) {           // torch rounds every NaN to the one with the first mantissa bit
#pragma unroll
                    for (int i = 0; i < VEC; ++i)
                        if (p[i] != p[i]) held[i] = __builtin_bit_cast(T, static_cast<Raw>(raw_bits<T>::INF | (raw_bits<T>::INF >> 1)));
                }
                if (prepared != nullptr) {
                    if constexpr (WHOLE) store_elems<T, VEC, SUM_NT>(prepared + e0[u], held);
                    else store_live<T, VEC, SUM_NT == kNonTemporal>(prepared + e0[u], valid - e0[u], held);
                }
            } else {
#pragma unroll
                for (int i = 0; i < VEC; ++i) held[i] = xv[u][i];
            }
            const int64_t group = e0[u] / G;
            const int k0 = static_cast<int>(e0[u] - group * G);
            float absmax;
            float multiplier = group_multiplier(m, absmax);   // every lane of the row takes part
            Raw stored = __builtin_bit_cast(Raw, narrow<T>(absmax));
            bool wide_codes = false;   // wavefront-uniform: codes may leave [-LEVELS, LEVELS]
            if (nans) {
                if (resets) {
                    const uint32_t scale_raw = scan_scale(held, group, k0);
                    multiplier = multiplier_of(value_of<T>(scale_raw));
                    stored = static_cast<Raw>(scale_raw);
                    wide_codes = true;
                } else {                            // fmaxf skips NaNs
                    uint32_t skipping = 0;
#pragma unroll
                    for (int i = 0; i < VEC; ++i) {
                        const uint32_t bits = as_u32(p[i]) & 0x7FFFFFFFu;
                        skipping = (bits <= 0x7F800000u && bits > skipping) ? bits : skipping;
                    }
                    multiplier = group_multiplier(skipping, absmax);
                    stored = __builtin_bit_cast(Raw, narrow<T>(absmax));
                }
            }
            int c[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) c[i] = cvt_i32(__builtin_rintf(p[i] * multiplier));
            if (wide_codes) clamp_codes(c);
            uint32_t words[W::WORDS];
            pack_codes<T, BIT, VEC, W::WORDS>(c, words);
            if (!WHOLE && e0[u] >= padded) continue;   // a lane's elements lie inside the padded range together
            // Interleaved 16-bit payloads leave as misaligned 8-byte stores here.  Re-slicing a pair of 66-byte groups
            // into aligned dwords across lanes (store_group_pair16, what the ring's gather hop does) measured slower in
            // this kernel at every size, with operands rotated through 700 MB: 26.2 M bf16 elements 15.8 us as it is,
            // 17.7 us with non-temporal pair stores, 16.1 us with cached ones; 52.4 M 27.4 / 32.8 / 27.6 us.  Nor does
            // it pay to stage a wavefront's run of eight groups (528 bytes, 16-byte aligned) in LDS and carry it out
            // as 33 aligned 16-byte stores: 16.2 us (16.4 us non-temporal) against 15.6 us on 26.2 M elements, no
            // workgroup barrier involved.  The misaligned stores are not what this layout costs.
            if constexpr (CODES == kWrittenThrough && WHOLE) {
                static_assert(CODES != kWrittenThrough || (!COMPACT && BIT == 8), "codes in the elements' order, a byte each");
                buffer_store<uint32_t, W::WORDS, kSc1Bit>(buffer_over(payload + block_first, BLOCK_ELEMS), static_cast<uint32_t>(e0[u] - block_first), words);
            } else {
                store_piece<T, BIT, CODES == kNonTemporal ? kNonTemporal : kPlain, W::WORDS>(payload + at.codes(group) + piece_offset<T, BIT>(k0), words);
            }
            if ((lane & (LPG - 1)) == 0) *reinterpret_cast<Raw *>(payload + at.scale(group)) = stored;
        }
    };
    if (block_first + BLOCK_ELEMS <= valid) tiles(std::true_type{});
    else tiles(std::false_type{});
}

template <typename T, int G, int BIT, bool HAS_R, bool COMPACT, int CODES, int TILES>
hipError_t launch_wire_quant_tiles(int mode, const WireQuantArgs &a, int world, hipStream_t stream) {
    constexpr int BLOCK_ELEMS = wire<T, BIT>::TILE * kWavesPerBlock * TILES;
    const int64_t groups = (a.shard_numel + G - 1) / G;
    const int64_t blocks = (groups * G + BLOCK_ELEMS - 1) / BLOCK_ELEMS;
    if (blocks == 0 || world == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL || world > 65535) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(world));
    if (mode == kStream) hipLaunchKernelGGL((wire_quant_kernel<T, G, BIT, HAS_R, COMPACT, kNonTemporal, CODES, TILES>), grid, dim3(kBlock), 0, stream, a);
    else hipLaunchKernelGGL((wire_quant_kernel<T, G, BIT, HAS_R, COMPACT, kPlain, kPlain, TILES>), grid, dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

// Tiles in flight per wavefront: one while they fit the chip's wavefront slots (us with one / four tiles: 10,048 fp32
// elements 1.9 / 2.6, 1 Mi 2.9 / 3.2, 2 Mi 3.5 / 4.0; bf16 10,048 2.0 / 2.5, 1 Mi 2.6 / 3.1, 4 Mi 3.7 / 4.4).  Beyond, two
// where a residual is read as well (13.1 M fp32 19.9 us, 20.7 with four; bf16 12.6 / 13.1), and without one four - for a
// 16-bit tensor two until there are twice the slots (6.6 M bf16 5.3 us with two, 6.0 with four; 13.1 M 9.3 / 9.1; fp32
// 6.6 M 7.8 / 7.6, 26.2 M 23.3 / 22.1).
template <typename T, int G, int BIT, bool HAS_R, bool COMPACT, int CODES>
hipError_t launch_wire_quant_s(int mode, const WireQuantArgs &a, int world, hipStream_t stream) {
    constexpr int64_t kOneEach = kResidentWaves * wire<T, BIT>::TILE;
    if (a.numel <= kOneEach) return launch_wire_quant_tiles<T, G, BIT, HAS_R, COMPACT, CODES, 1>(mode, a, world, stream);
    if constexpr (HAS_R) {
        return launch_wire_quant_tiles<T, G, BIT, HAS_R, COMPACT, CODES, 2>(mode, a, world, stream);
    } else {
        if constexpr (sizeof(T) == 2) {
            if (a.numel <= 2 * kOneEach) return launch_wire_quant_tiles<T, G, BIT, HAS_R, COMPACT, CODES, 2>(mode, a, world, stream);
        }
        return launch_wire_quant_tiles<T, G, BIT, HAS_R, COMPACT, CODES, 4>(mode, a, world, stream);
    }
}

// How the codes leave.  Interleaved with the scales in plain stores (a line is shared by neighbouring wavefronts).  Apart
// from them with the non-temporal hint where they leave for other ranks (chunks), and for small tensors; the one payload of a large
// tensor is read by its decode, or by a reduce, next.  us of quantize + decode, non-temporal / plain / written through, three
// tensors in rotation and (in brackets) enough of them to outrun the last-level cache: fp32 4.3 M 11.5 / 11.0 / 10.4 (11.6 /
// 10.5 / 10.8), 6.6 M 15.4 / 14.7 / 14.2 (15.3 / 13.6 / 14.0), 13.1 M 26.8 / 26.1 / 24.0 (25.6 / 23.1 / 23.1), 26.2 M 46.0 / 42.0 /
// 42.4 (45.3 / 41.3 / 41.1), 52.4 M 85.6 / 79.0 / 77.3 (85.9 / 79.2 / 77.5); with the reduce of two payloads as the reader 6.6 M
// 16.3 / 15.4 / 15.4, 13.1 M 28.5 / 27.0 / 26.1, 26.2 M 49.5 / 45.3 / 45.1, of four and eight 2 % slower at 6.6 M (18.9 / 19.3 / 19.3,
// 23.6 / 23.7 / 24.1) and 2 % faster at 26.2 M.  16-bit, non-temporal / plain, decode and reduce of two: 8.4 M 13.8 / 14.2 and
// 15.0 / 15.6 (14.0 / 12.4 and 16.1 / 15.5), 13.1 M 19.0 / 19.3 and 19.7 / 20.3 (18.5 / 16.1 and 20.0 / 19.2), 14.7 M 22.3 / 21.0 and
// 20.9 / 21.3, 16.8 M 23.3 / 23.3 and 23.7 / 23.5 (22.9 / 20.0 and 24.9 / 23.8), 26.2 M 31.4 / 29.3 and 33.0 / 31.9: up to 7 %
// slower in rotation below the line, faster on both sides of the cache from it on.  4-bit codes keep the hint (26.2 M 41.5 / 41.5 and
// 27.3 / 28.0).  Beside a residual plain at every size (SUM_NT above; the hook's two launches, 2.5 M fp32 of two payloads 14.8 ->
// 11.6 us, of eight 16.5 -> 15.9, 26.2 M 113.5 -> 104.8 and 140.9 -> 132.4; four payloads of 4.3 and 9.0 M 2 % slower).
template <typename T, int G, int BIT, bool HAS_R, bool COMPACT>
hipError_t launch_wire_quant_c(int mode, const WireQuantArgs &a, int world, hipStream_t stream) {
    if constexpr (COMPACT) return launch_wire_quant_s<T, G, BIT, HAS_R, COMPACT, kPlain>(mode, a, world, stream);
    if constexpr (HAS_R && !COMPACT) {
        if (world == 1) return launch_wire_quant_s<T, G, BIT, HAS_R, COMPACT, kPlain>(mode, a, world, stream);
    } else if constexpr (BIT == 8 && !COMPACT) {
        constexpr int64_t kLarge = (sizeof(T) == 4 ? int64_t{4} : int64_t{16}) << 20;
        constexpr int KEPT = sizeof(T) == 4 ? kWrittenThrough : kPlain;
        if (world == 1 && a.numel > kLarge) return launch_wire_quant_tiles<T, G, BIT, HAS_R, COMPACT, KEPT, 4>(mode, a, world, stream);
    }
    return launch_wire_quant_s<T, G, BIT, HAS_R, COMPACT, kNonTemporal>(mode, a, world, stream);
}

template <typename T, int G, int BIT>
hipError_t launch_wire_quant_b(int mode, const WireQuantArgs &a, int world, hipStream_t stream) {
    if (a.residual != nullptr)
        return a.compact ? launch_wire_quant_c<T, G, BIT, true, true>(mode, a, world, stream)
                         : launch_wire_quant_c<T, G, BIT, true, false>(mode, a, world, stream);
    return a.compact ? launch_wire_quant_c<T, G, BIT, false, true>(mode, a, world, stream)
                     : launch_wire_quant_c<T, G, BIT, false, false>(mode, a, world, stream);
}

template <typename T, int G>
hipError_t launch_wire_quant_g(int bit, int mode, const WireQuantArgs &a, int world, hipStream_t stream) {
    if (bit == 8) return launch_wire_quant_b<T, G, 8>(mode, a, world, stream);
    if (bit == 4) return launch_wire_quant_b<T, G, 4>(mode, a, world, stream);
    return hipErrorNotSupported;
}

template <typename T>
hipError_t launch_wire_quant_t(int g, int bit, int mode, const WireQuantArgs &a, int world, hipStream_t s) {
    switch (g) {
        case 64: return launch_wire_quant_g<T, 64>(bit, mode, a, world, s);
        case 32: return launch_wire_quant_g<T, 32>(bit, mode, a, world, s);
        case 16: return launch_wire_quant_g<T, 16>(bit, mode, a, world, s);
        default: return hipErrorNotSupported;
    }
}

// ---------------------------------------------------------------------------
// fused dequant-reduce of up to 8 payloads (+ mean, + error-feedback update)
// ---------------------------------------------------------------------------
// Buffer stores go to 16-byte aligned tensors only; everything else here takes any element.
bool whole_vectors(const void *a, const void *b = nullptr) {
    return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0;
}

// KEPT: whole blocks write their outputs through the L2 without the non-temporal hint and load `prepared` with the codes; the
// launcher says when.
template <typename T, int G, int WORLD, bool FMA, bool COMPACT, int NT, bool WINDOWS = false, bool KEPT = false>
__global__ __launch_bounds__(kBlock) void wire_reduce_kernel(const WireReduceArgs a) {
    constexpr int PNT = payload_load_hint<COMPACT, NT, WORLD>();
    using W = wire<T>;
    constexpr int VEC = W::VEC;
    constexpr int UNROLL = WORLD <= 2 ? 2 : 1;
    constexpr int BLOCK_ELEMS = W::TILE * kWavesPerBlock * UNROLL;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(BLOCK_ELEMS)) * BLOCK_ELEMS;
    const int64_t groups = (a.numel + G - 1) / G;
    const group_layout<T, G, COMPACT> at{groups};
    T *__restrict__ out = static_cast<T *>(a.out);
    const T *prepared = static_cast<const T *>(a.prepared);  // may alias new_r
    T *new_r = static_cast<T *>(a.new_residual);

    auto store_whole = [&](T *base, int64_t e, const T (&v)[VEC]) __attribute__((always_inline)) {
        if constexpr (KEPT) buffer_store<T, VEC, kSc1Bit>(buffer_over(base + block_first, BLOCK_ELEMS * sizeof(T)), static_cast<uint32_t>(e - block_first) * sizeof(T), v);
        else store_elems<T, VEC, NT>(base + e, v);
    };
    auto accumulate = [](float acc, float code, float step) {
        if constexpr (FMA) return __builtin_fmaf(code, step, acc);
        else return acc + code * step;
    };

    // One pass over the block's tiles, the codes and scales of all of them issued before the arithmetic (`prepared` with
    // them in the last block; whole blocks load it tile by tile, after the decode).  WHOLE: all of the block's outputs
    // exist; otherwise a lane's vector is cut short at the end (the payload holds whole groups, so a lane with one live
    // output may read all of its codes).  Element by element the last block was the longest chain of a
    // mid-sized launch: 10,048 outputs of eight payloads, interleaved bf16 4.2 us then, 2.4 now, fp32 with error feedback
    // 3.7 and 2.2, 2 Mi of two bf16 payloads with error feedback 5.1 and 4.9; decode of 10,048 2.9 and 1.9.
    auto tiles = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        uint32_t words[UNROLL][WORLD][W::WORDS];
        T stored[UNROLL][WORLD];
        T pv[UNROLL][VEC];
        int64_t e0[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            e0[u] = block_first + static_cast<int64_t>(tile_in_block<UNROLL>(u, wave)) * W::TILE + lane * VEC;
            const int64_t group = e0[u] / G;
            const int k0 = static_cast<int>(e0[u] - group * G);
            const int64_t code_at = at.codes(group) + k0;
            const int64_t scale_at = at.scale(group);
            if constexpr (WINDOWS) {   // 16-bit compact payloads below 2 GiB: aligned windows, scales out of them;
                static_assert(COMPACT && sizeof(T) == 2 && G == 64 && W::WORDS == 2, "66-byte groups of 8 lanes");
                const uint32_t payload_bytes = static_cast<uint32_t>(groups * (G + 2));   // past the payload: zeros
#pragma unroll
                for (int r = 0; r < WORLD; ++r) {
                    const uint32_t lead = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(a.payloads[r]) & 3u);
                    uint32_t after;
                    load_piece16<window_policy<NT, WORLD>()>(buffer_over(a.payloads[r] - lead, window_span(payload_bytes + lead)),
                                          static_cast<uint32_t>(WHOLE || e0[u] < groups * G ? code_at : 0) + lead, words[u][r], after);
                    const uint32_t raw = from_last_lane_of_8(after, (lane & 8) != 0);
                    stored[u][r] = __builtin_bit_cast(T, static_cast<uint16_t>(raw));
                }
            } else {
#pragma unroll
                for (int r = 0; r < WORLD; ++r) {
#pragma unroll
                    for (int k = 0; k < W::WORDS; ++k) words[u][r][k] = 0;
                    stored[u][r] = narrow<T>(0.0f);
                    if (WHOLE || e0[u] < a.numel) {
                        load_words<W::WORDS, sizeof(T), PNT>(a.payloads[r] + code_at, words[u][r]);
                        stored[u][r] = *reinterpret_cast<const T *>(a.payloads[r] + scale_at);
                    }
                }
            }
            if (new_r != nullptr) {
                if constexpr (WHOLE && KEPT) load_elems<T, VEC, NT>(prepared + e0[u], pv[u]);
                else if constexpr (!WHOLE) load_live<T, VEC, NT == kNonTemporal>(prepared + e0[u], a.numel - e0[u], pv[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            float acc[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = 0.0f;
#pragma unroll
            for (int r = 0; r < WORLD; ++r) {
                const float step = div127(widen(stored[u][r]));
#pragma unroll
                for (int i = 0; i < VEC; ++i)
                    acc[i] = accumulate(acc[i], code_to_float(words[u][r][i / 4], byte_in_word<T>(i % 4)), step);
            }
            T o[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = acc[i] * a.inv_divisor;
            narrow_all<T, VEC>(acc, o);
            if constexpr (WHOLE) store_whole(out, e0[u], o);
            else store_live<T, VEC, NT == kNonTemporal>(out + e0[u], a.numel - e0[u], o);
            if (new_r != nullptr) {
                T d[VEC];
                float left[VEC];
                if constexpr (WHOLE && !KEPT) load_elems<T, VEC, NT>(prepared + e0[u], pv[u]);
#pragma unroll
                for (int i = 0; i < VEC; ++i) left[i] = widen(pv[u][i]) - acc[i];
                narrow_all<T, VEC>(left, d);
                if constexpr (WHOLE) store_whole(new_r, e0[u], d);
                else store_live<T, VEC, NT == kNonTemporal>(new_r + e0[u], a.numel - e0[u], d);
            }
        }
    };
    if (block_first + BLOCK_ELEMS <= a.numel) tiles(std::true_type{});
    else tiles(std::false_type{});
}

template <typename T, int G, int WORLD, bool FMA, bool COMPACT>
hipError_t launch_wire_reduce_c(int mode, const WireReduceArgs &a, hipStream_t stream) {
    constexpr int BLOCK_ELEMS = wire<T>::TILE * kWavesPerBlock * (WORLD <= 2 ? 2 : 1);
    const int64_t blocks = (a.numel + BLOCK_ELEMS - 1) / BLOCK_ELEMS;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    if constexpr (COMPACT && sizeof(T) == 2) {
        if ((a.numel + G - 1) / G * (G + 2) < (1LL << 31)) {   // a buffer descriptor spans the payload
            if (mode == kStream) hipLaunchKernelGGL((wire_reduce_kernel<T, G, WORLD, FMA, COMPACT, kNonTemporal, true>), grid, dim3(kBlock), 0, stream, a);
            else hipLaunchKernelGGL((wire_reduce_kernel<T, G, WORLD, FMA, COMPACT, kPlain, true>), grid, dim3(kBlock), 0, stream, a);
            return hipGetLastError();
        }
    }
    // KEPT: scales apart, four payloads or more, with feedback, and an output of a size that gains in rotation and does not lose
    // beyond the last-level cache, where a training run's buckets are.  GPU us of the hook's two launches, non-temporal / KEPT, three
    // states in rotation (and beyond the cache): eight payloads fp32 1 MiB 4.87 / 4.55 (5.99 / 5.66), 12 MiB 21.9 / 20.4 (21.7 / 21.3),
    // 25 MiB 38.9 / 37.2 (38.4 / 38.1), 40 MiB 58.6 / 56.9 (57.8 / 58.5); bf16 0.8 MiB 6.3 / 6.0 (8.6 / 8.4), 15 MiB 31.1 / 29.7 (30.9 /
    // 30.9), 24 MiB 49.3 / 48.0 (48.0 / 48.6); four bf16 0.1 MiB 5.2 / 5.2 (6.0 / 6.2), 30 MiB 47.6 / 44.9 (47.2 / 46.5).  Four fp32 of 2
    // to 8 MiB lose either way, 7 MiB 11.1 / 12.2 (11.8 / 12.9).  Without feedback it loses beyond the cache (eight fp32 32 MiB 26.1 / 25.9
    // (25.8 / 26.9)), with two payloads as well (fp32 6.6 M elements 29.9 / 34.1), with interleaved scales everywhere.
    if constexpr (!COMPACT && WORLD >= 4) {
        const int64_t kib = (a.numel * static_cast<int64_t>(sizeof(T)) + 1023) >> 10;
        const bool gains = sizeof(T) == 2 ? kib >= 256 && kib < (WORLD <= 6 ? 32 << 10 : 16 << 10)
                                          : kib <= 1536 || (kib >= 9 << 10 && kib < 32 << 10);
        if (mode == kStream && a.new_residual != nullptr && gains && whole_vectors(a.out, a.new_residual)) {
            hipLaunchKernelGGL((wire_reduce_kernel<T, G, WORLD, FMA, COMPACT, kNonTemporal, false, true>), grid, dim3(kBlock), 0, stream, a);
            return hipGetLastError();
        }
    }
    if (mode == kStream) hipLaunchKernelGGL((wire_reduce_kernel<T, G, WORLD, FMA, COMPACT, kNonTemporal>), grid, dim3(kBlock), 0, stream, a);
    else hipLaunchKernelGGL((wire_reduce_kernel<T, G, WORLD, FMA, COMPACT, kPlain>), grid, dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

template <typename T, int G, int WORLD, bool FMA>
hipError_t launch_wire_reduce_w(int mode, const WireReduceArgs &a, hipStream_t stream) {
    return a.compact ? launch_wire_reduce_c<T, G, WORLD, FMA, true>(mode, a, stream)
                     : launch_wire_reduce_c<T, G, WORLD, FMA, false>(mode, a, stream);
}

template <typename T, int G, bool FMA>
hipError_t launch_wire_reduce_f(int world, int mode, const WireReduceArgs &a, hipStream_t s) {
    switch (world) {
        case 1: return launch_wire_reduce_w<T, G, 1, FMA>(mode, a, s);
        case 2: return launch_wire_reduce_w<T, G, 2, FMA>(mode, a, s);
        case 3: return launch_wire_reduce_w<T, G, 3, FMA>(mode, a, s);
        case 4: return launch_wire_reduce_w<T, G, 4, FMA>(mode, a, s);
        case 5: return launch_wire_reduce_w<T, G, 5, FMA>(mode, a, s);
        case 6: return launch_wire_reduce_w<T, G, 6, FMA>(mode, a, s);
        case 7: return launch_wire_reduce_w<T, G, 7, FMA>(mode, a, s);
        case 8: return launch_wire_reduce_w<T, G, 8, FMA>(mode, a, s);
        default: return hipErrorNotSupported;
    }
}

template <typename T>
hipError_t launch_wire_reduce_t(int g, int world, bool fma, int mode, const WireReduceArgs &a, hipStream_t s) {
    if (g != 64) return hipErrorNotSupported;   // as the reference: dequant_reduce_kernel.cu:17,252
    return fma ? launch_wire_reduce_f<T, 64, true>(world, mode, a, s) : launch_wire_reduce_f<T, 64, false>(world, mode, a, s);
}

// ---------------------------------------------------------------------------
// decode of one payload (optionally combined into `out`), or of `world` shard payloads
// ---------------------------------------------------------------------------
template <typename T, int OP> __device__ __forceinline__ float combine_in(float old, float v) {
    if constexpr (OP == 1) return add_in<T>(old, v);
    else if constexpr (OP == 2) return old > v ? old : v;
    else if constexpr (OP == 3) return old > v ? v : old;
    else return v;
}

// THROUGH: whole blocks write their outputs through the L2 beside the non-temporal hint.
template <typename T, int G, int BIT, int OP, bool COMPACT, int NT, bool THROUGH = false>
__global__ __launch_bounds__(kBlock) void wire_decode_kernel(const WireDecodeArgs a) {
    constexpr int PNT = payload_load_hint<COMPACT, NT, 1>();
    using W = wire<T, BIT>;
    constexpr int VEC = W::VEC;
    constexpr int UNROLL = 2;
    constexpr int BLOCK_ELEMS = W::TILE * kWavesPerBlock * UNROLL;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t chunk = blockIdx.y;
    const int64_t chunk_start = chunk * a.shard_numel;
    int64_t valid = a.total_numel - chunk_start;
    valid = valid < 0 ? 0 : (valid > a.shard_numel ? a.shard_numel : valid);
    const int64_t groups = (a.shard_numel + G - 1) / G;
    const group_layout<T, G, COMPACT, BIT> at{groups};
    const uint8_t *__restrict__ payload = a.payloads + chunk * a.payload_stride;
    T *__restrict__ out = static_cast<T *>(a.out) + chunk_start;
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(BLOCK_ELEMS)) * BLOCK_ELEMS;
    if (block_first >= valid) return;

    auto tiles = [&](auto whole) __attribute__((always_inline)) {   // WHOLE as in the reduce
        constexpr bool WHOLE = decltype(whole)::value;
        uint32_t words[UNROLL][W::WORDS];
        T stored[UNROLL];
        T o[UNROLL][VEC];
        int64_t e0[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            e0[u] = block_first + static_cast<int64_t>(tile_in_block<UNROLL>(u, wave)) * W::TILE + lane * VEC;
            const int64_t group = e0[u] / G;
            const int k0 = static_cast<int>(e0[u] - group * G);
#pragma unroll
            for (int k = 0; k < W::WORDS; ++k) words[u][k] = 0;
            stored[u] = narrow<T>(0.0f);
            if (WHOLE || e0[u] < valid) {
                load_piece<T, BIT, PNT, W::WORDS>(payload + at.codes(group) + piece_offset<T, BIT>(k0), words[u]);
                stored[u] = *reinterpret_cast<const T *>(payload + at.scale(group));
            }
            if constexpr (OP != 0 && !WHOLE) load_live<T, VEC, NT == kNonTemporal>(out + e0[u], valid - e0[u], o[u]);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            if constexpr (OP != 0 && WHOLE) load_elems<T, VEC, NT>(out + e0[u], o[u]);
            const float step = step_of<BIT>(widen(stored[u]));
            float v[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) v[i] = unpack_code<T, BIT, W::WORDS>(words[u], i) * step;
            if constexpr (OP != 0) {
                round_through_all<T, VEC>(v);
#pragma unroll
                for (int i = 0; i < VEC; ++i) v[i] = combine_in<T, OP>(widen(o[u][i]), v[i]);
            }
            narrow_all<T, VEC>(v, o[u]);
            if constexpr (WHOLE && THROUGH) buffer_store<T, VEC, kNtBit | kSc1Bit>(buffer_over(out + block_first, BLOCK_ELEMS * sizeof(T)), static_cast<uint32_t>(e0[u] - block_first) * sizeof(T), o[u]);
            else if constexpr (WHOLE) store_elems<T, VEC, NT>(out + e0[u], o[u]);
            else store_live<T, VEC, NT == kNonTemporal>(out + e0[u], valid - e0[u], o[u]);
        }
    };
    if (block_first + BLOCK_ELEMS <= valid) tiles(std::true_type{});
    else tiles(std::false_type{});
}

template <typename T, int G, int BIT, int OP, bool COMPACT>
hipError_t launch_wire_decode_c(int mode, const WireDecodeArgs &a, int world, hipStream_t stream) {
    constexpr int BLOCK_ELEMS = wire<T, BIT>::TILE * kWavesPerBlock * 2;
    const int64_t blocks = (a.shard_numel + BLOCK_ELEMS - 1) / BLOCK_ELEMS;
    if (blocks == 0 || world == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL || world > 65535) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(world));
    // One payload: THROUGH from 16 MiB of outputs on, 8-bit fp32 ones from 32 MiB on.  us of quantize + decode, nt alone / both, three
    // tensors in rotation (and beyond the last-level cache): bf16 16 MiB 13.7 / 13.3 (13.6 / 13.4), 25 MiB 18.5 / 17.9 (18.7 / 18.2),
    // interleaved 25 MiB 16.4 / 16.2 (16.8 / 16.6), 4-bit 25 MiB 16.9 / 16.1 (16.0 / 15.8), 1 Mi elements 4.50 / 4.40 (4.9 / 5.3); fp32 20 MiB 12.2 /
    // 12.1 (11.9 / 12.0), interleaved 12.3 / 12.0 (11.7 / 11.8), 4-bit 11.8 / 11.7 (11.4 / 11.4), 25 MiB 14.5 / 14.4 (14.1 / 14.2), 32 MiB 16.5 / 16.3
    // (16.4 / 16.4), 100 MiB 41.5 / 41.4 (41.3 / 41.2), 4-bit 39.4 / 38.5 (38.9 / 38.1).
    if constexpr (OP == 0) {
        constexpr int64_t kThrough = int64_t{sizeof(T) == 2 || BIT == 4 ? 16 : 32} << 20;
        if (mode == kStream && world == 1 && whole_vectors(a.out) && a.total_numel * static_cast<int64_t>(sizeof(T)) >= kThrough) {
            hipLaunchKernelGGL((wire_decode_kernel<T, G, BIT, OP, COMPACT, kNonTemporal, true>), grid, dim3(kBlock), 0, stream, a);
            return hipGetLastError();
        }
    }
    if (mode == kStream) hipLaunchKernelGGL((wire_decode_kernel<T, G, BIT, OP, COMPACT, kNonTemporal>), grid, dim3(kBlock), 0, stream, a);
    else hipLaunchKernelGGL((wire_decode_kernel<T, G, BIT, OP, COMPACT, kPlain>), grid, dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

template <typename T, int G, int BIT, int OP>
hipError_t launch_wire_decode_op(int mode, const WireDecodeArgs &a, int world, hipStream_t stream) {
    return a.compact ? launch_wire_decode_c<T, G, BIT, OP, true>(mode, a, world, stream)
                     : launch_wire_decode_c<T, G, BIT, OP, false>(mode, a, world, stream);
}

template <typename T, int G, int BIT>
hipError_t launch_wire_decode_b(int op, int mode, const WireDecodeArgs &a, int world, hipStream_t s) {
    switch (op) {
        case 0: return launch_wire_decode_op<T, G, BIT, 0>(mode, a, world, s);
        case 1: return launch_wire_decode_op<T, G, BIT, 1>(mode, a, world, s);
        case 2: return launch_wire_decode_op<T, G, BIT, 2>(mode, a, world, s);
        case 3: return launch_wire_decode_op<T, G, BIT, 3>(mode, a, world, s);
        default: return hipErrorNotSupported;
    }
}

template <typename T, int G>
hipError_t launch_wire_decode_g(int bit, int op, int mode, const WireDecodeArgs &a, int world, hipStream_t s) {
    if (bit == 8) return launch_wire_decode_b<T, G, 8>(op, mode, a, world, s);
    if (bit == 4) return launch_wire_decode_b<T, G, 4>(op, mode, a, world, s);
    return hipErrorNotSupported;
}

template <typename T>
hipError_t launch_wire_decode_t(int g, int bit, int op, int mode, const WireDecodeArgs &a, int world, hipStream_t s) {
    switch (g) {
        case 64: return launch_wire_decode_g<T, 64>(bit, op, mode, a, world, s);
        case 32: return launch_wire_decode_g<T, 32>(bit, op, mode, a, world, s);
        case 16: return launch_wire_decode_g<T, 16>(bit, op, mode, a, world, s);
        default: return hipErrorNotSupported;
    }
}

// ---------------------------------------------------------------------------
// ring / tree step in this format: chunk (op)= decode(received) [* 1/W], then the quantize of the updated chunk
// ---------------------------------------------------------------------------
// What a rank running the reference does per hop with its extension loaded (torch_topology.py:262-316): decode the
// arriving payload into the chunk with reduce op SUM or NONE, `div_` by the world size on the hop that completes
// the sum (a multiplication by the float reciprocal, the way torch divides a device tensor by a number), then
// quantize the chunk for the next hop - here in one launch, the updated chunk still in registers.  Linear 8-bit
// codes, whole groups (the reference's in-place decode needs them).  The encode is the one a chunk of whole groups
// without a residual gets in the reference: group maximum with NaNs skipped, and when a group holds a NaN the
// running maximum of the general kernels, which a NaN resets (see wire_quant_kernel).
template <typename T, bool ACC> constexpr int wire_ring_unroll() { return ACC || sizeof(T) == 2 ? 1 : 4; }

template <typename T, int G, bool COMPACT, int NT, bool ACC, bool WINDOWS = false>
__global__ __launch_bounds__(kBlock) void wire_ring_step_kernel(const WireRingStepArgs a) {
    constexpr int PNT_LOAD = payload_load_hint<COMPACT, NT, 1>();
    constexpr int PNT_STORE = COMPACT ? kPlain : NT;
    using W = wire<T, 8>;
    using Raw = typename raw_bits<T>::type;
    constexpr int VEC = W::VEC;
    constexpr int LPG = G / VEC;
    // Tiles in flight per wavefront, as measured on 6.5 M to 52 M element chunks: one for the accumulating step and
    // for 16-bit chunks, four for the write-only steps on fp32 chunks.
    constexpr int UNROLL = wire_ring_unroll<T, ACC>();
    constexpr int BLOCK_ELEMS = W::TILE * kWavesPerBlock * UNROLL;
    static_assert(LPG >= 1 && LPG <= 16, "a group must fit one DPP row");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t groups = a.numel / G;               // whole groups only
    const group_layout<T, G, COMPACT, 8> at{groups};
    const uint8_t *__restrict__ received = a.received;
    T *chunk = static_cast<T *>(a.chunk);
    const bool scaled = a.inv_divisor != 1.0f;
    const bool emit = a.send != nullptr;
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(BLOCK_ELEMS)) * BLOCK_ELEMS;
    if (block_first >= a.numel) return;

    uint32_t words[UNROLL][W::WORDS];
    T stored[UNROLL];
    T xv[UNROLL][VEC];
    int64_t e0[UNROLL];
    bool live[UNROLL];   // a lane's elements, and its whole group, lie inside the chunk or outside it together
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
        e0[u] = block_first + static_cast<int64_t>(tile_in_block<UNROLL>(u, wave)) * W::TILE + lane * VEC;
        live[u] = e0[u] < a.numel;
        if constexpr (WINDOWS) {   // 16-bit compact payload below 2 GiB: aligned windows, the scale out of them;
            static_assert(COMPACT && sizeof(T) == 2 && G == 64 && W::WORDS == 2, "66-byte groups of 8 lanes");
            const int64_t group = e0[u] / G;                    // a window past the payload reads as zeros
            const int k0 = static_cast<int>(e0[u] - group * G);
            const uint32_t lead = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(received) & 3u);
            uint32_t after;
            load_piece16<window_policy<NT, 1>()>(buffer_over(received - lead, window_span(static_cast<uint32_t>(groups * (G + 2)) + lead)),
                                                 static_cast<uint32_t>(live[u] ? at.codes(group) + k0 : 0) + lead, words[u], after);
            stored[u] = __builtin_bit_cast(T, static_cast<uint16_t>(from_last_lane_of_8(after, (lane & 8) != 0)));
            if constexpr (ACC) {
                if (live[u]) load_elems<T, VEC, NT>(chunk + e0[u], xv[u]);
            }
        } else if (live[u]) {
            const int64_t group = e0[u] / G;
            const int k0 = static_cast<int>(e0[u] - group * G);
            load_piece<T, 8, PNT_LOAD, W::WORDS>(received + at.codes(group) + piece_offset<T, 8>(k0), words[u]);
            stored[u] = *reinterpret_cast<const T *>(received + at.scale(group));
            if constexpr (ACC) load_elems<T, VEC, NT>(chunk + e0[u], xv[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
        float p[VEC];
        T held[VEC];
        uint32_t m = 0;   // largest magnitude pattern; above the pattern of infinity when the lane holds a NaN
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            p[i] = 0.0f;
            held[i] = narrow<T>(0.0f);
        }
        if (live[u]) {
            const float step = step_of<8>(widen(stored[u]));
#pragma unroll
            for (int i = 0; i < VEC; ++i) p[i] = unpack_code<T, 8, W::WORDS>(words[u], i) * step;
            round_through_all<T, VEC>(p);
            if constexpr (ACC) {
#pragma unroll
                for (int i = 0; i < VEC; ++i) p[i] = widen(xv[u][i]) + p[i];
                round_through_all<T, VEC>(p);
            }
            if (scaled) {
#pragma unroll
                for (int i = 0; i < VEC; ++i) p[i] = p[i] * a.inv_divisor;
                round_through_all<T, VEC>(p);
            }
            narrow_all<T, VEC>(p, held);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const uint32_t bits = as_u32(p[i]) & 0x7FFFFFFFu;
                m = bits > m ? bits : m;
            }
            store_elems<T, VEC, NT>(chunk + e0[u], held);
        }
        if (!emit) continue;    // uniform over the grid
        // every lane of a row takes part in the group reductions; rows past the end carry zeros
        const int64_t group = e0[u] / G;
        const int k0 = static_cast<int>(e0[u] - group * G);
        const float absmax = as_f32(group_max_bits<LPG>(m));   // the group maximum when the wavefront holds no NaN
        float scale = absmax < 1.0e-6f ? 1.0e-6f : absmax;
        Raw kept = __builtin_bit_cast(Raw, narrow<T>(absmax));
        bool wide_codes = false;                               // wavefront-uniform
        if (__ballot(m > 0x7F800000u) != 0) {                  // a NaN somewhere: every group is scanned again
            uint32_t mag[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) mag[i] = __builtin_bit_cast(Raw, held[i]) & raw_bits<T>::ABS;
            const uint32_t scale_raw = running_max_raw<T, G, VEC>(mag, k0, scan_start<T, G>(group));
            const float rescanned = value_of<T>(scale_raw);
            scale = rescanned < 1.0e-6f ? 1.0e-6f : rescanned;
            kept = static_cast<Raw>(scale_raw);
            wide_codes = true;
        }
        const float multiplier = W::LEVELS / scale;
        int c[VEC];
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            c[i] = cvt_i32(__builtin_rintf(p[i] * multiplier));
            if (wide_codes) c[i] = c[i] < -127 ? -127 : (c[i] > 127 ? 127 : c[i]);
        }
        uint32_t out_words[W::WORDS];
        pack_codes<T, 8, VEC, W::WORDS>(c, out_words);
        if constexpr (WINDOWS) {
            // The hop that only decodes and requantizes, from 4 Mi elements on (uniform): the payload leaves as
            // whole dwords shifted across lanes, with the non-temporal hint.  Measured with operands rotated through
            // 700 MB, bf16: 52 M elements 38.8 instead of 43.3 us, 26 M 19.8 instead of 21.5, 13.1 M 11.4 instead
            // of 12.9, 6.5 M 7.3 instead of 8.3; 3.3 M 6.3 against 5.3 and 1.6 M 4.5 either way, hence the bound.
            // (With only a few buffer sets, i.e. payloads that stay in the last-level cache, 13.1 M read 11.4
            // against 10.9 us, which is where an earlier bound of 16 Mi came from.)  Both forms write exactly the
            // chunk and the payload (rocprofv3 WRITE_SIZE 38,800 KiB against 39,082 KiB on 13.1 M elements) and read
            // exactly the payload: the gain is in the store instructions, not in traffic.  The accumulating hop and
            // the quantize kernel lost 1-20 % with the same stores.
            if ((reinterpret_cast<uintptr_t>(a.send) & 3u) == 0 && a.numel >= (int64_t{1} << LBC_PAIR_STORE_MIN_LOG2)) {
                store_group_pair16<kNonTemporal>(a.send + at.codes(group & ~int64_t{1}), lane, out_words, kept, live[u],
                                              (group | 1) < groups);
                continue;
            }
        }
        if (!live[u]) continue;
        store_piece<T, 8, PNT_STORE, W::WORDS>(a.send + at.codes(group) + piece_offset<T, 8>(k0), out_words);
        if ((lane & (LPG - 1)) == 0) *reinterpret_cast<Raw *>(a.send + at.scale(group)) = kept;
    }
}

template <typename T, int G, bool COMPACT, bool ACC>
hipError_t launch_wire_ring_c(int mode, const WireRingStepArgs &a, hipStream_t stream) {
    constexpr int BLOCK_ELEMS = wire<T, 8>::TILE * kWavesPerBlock * wire_ring_unroll<T, ACC>();
    const int64_t blocks = (a.numel + BLOCK_ELEMS - 1) / BLOCK_ELEMS;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    // Aligned windows for the received payload pay on the hop that only decodes and requantizes (52 M bf16
    // elements: 43 against 47.5 us); on the accumulating hop, where the chunk is read as well, they measured 2 %
    // slower, and a single-payload decode does not notice them (the payload is a third of its traffic).
    if constexpr (COMPACT && sizeof(T) == 2 && G == 64 && !ACC) {
        if (a.numel / G * (G + 2) < (1LL << 31)) {   // a buffer descriptor spans the payload
            if (mode == kStream) hipLaunchKernelGGL((wire_ring_step_kernel<T, G, COMPACT, kNonTemporal, ACC, true>), grid, dim3(kBlock), 0, stream, a);
            else hipLaunchKernelGGL((wire_ring_step_kernel<T, G, COMPACT, kPlain, ACC, true>), grid, dim3(kBlock), 0, stream, a);
            return hipGetLastError();
        }
    }
    if (mode == kStream) hipLaunchKernelGGL((wire_ring_step_kernel<T, G, COMPACT, kNonTemporal, ACC>), grid, dim3(kBlock), 0, stream, a);
    else hipLaunchKernelGGL((wire_ring_step_kernel<T, G, COMPACT, kPlain, ACC>), grid, dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

template <typename T, int G>
hipError_t launch_wire_ring_g(bool accumulate, int mode, const WireRingStepArgs &a, hipStream_t s) {
    if (a.compact) return accumulate ? launch_wire_ring_c<T, G, true, true>(mode, a, s) : launch_wire_ring_c<T, G, true, false>(mode, a, s);
    return accumulate ? launch_wire_ring_c<T, G, false, true>(mode, a, s) : launch_wire_ring_c<T, G, false, false>(mode, a, s);
}

template <typename T>
hipError_t launch_wire_ring_t(int g, bool accumulate, int mode, const WireRingStepArgs &a, hipStream_t s) {
    switch (g) {
        case 64: return launch_wire_ring_g<T, 64>(accumulate, mode, a, s);
        case 32: return launch_wire_ring_g<T, 32>(accumulate, mode, a, s);
        case 16: return launch_wire_ring_g<T, 16>(accumulate, mode, a, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace

hipError_t launch_wire_quant(int dtype, int group_size, int bit, int mode, const WireQuantArgs &args, int world,
                             hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_wire_quant_t<float>(group_size, bit, mode, args, world, stream);
        case kF16: return launch_wire_quant_t<f16>(group_size, bit, mode, args, world, stream);
        case kBF16: return launch_wire_quant_t<bf16>(group_size, bit, mode, args, world, stream);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_wire_reduce(int dtype, int group_size, int world, bool fused_multiply_add, int mode,
                              const WireReduceArgs &args, hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_wire_reduce_t<float>(group_size, world, fused_multiply_add, mode, args, stream);
        case kF16: return launch_wire_reduce_t<f16>(group_size, world, fused_multiply_add, mode, args, stream);
        case kBF16: return launch_wire_reduce_t<bf16>(group_size, world, fused_multiply_add, mode, args, stream);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_wire_decode(int dtype, int group_size, int bit, int reduce_op, int mode, const WireDecodeArgs &args,
                              int world, hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_wire_decode_t<float>(group_size, bit, reduce_op, mode, args, world, stream);
        case kF16: return launch_wire_decode_t<f16>(group_size, bit, reduce_op, mode, args, world, stream);
        case kBF16: return launch_wire_decode_t<bf16>(group_size, bit, reduce_op, mode, args, world, stream);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_wire_ring_step(int dtype, int group_size, bool accumulate, int mode, const WireRingStepArgs &args,
                                 hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_wire_ring_t<float>(group_size, accumulate, mode, args, stream);
        case kF16: return launch_wire_ring_t<f16>(group_size, accumulate, mode, args, stream);
        case kBF16: return launch_wire_ring_t<bf16>(group_size, accumulate, mode, args, stream);
        default: return hipErrorNotSupported;
    }
}

}  // namespace lbc
