// Device side of quantize + pack: what one workgroup does.  Shared by the quantize kernel and by the kernel that
// carries a quantize and a fused reduce in one grid.
#pragma once

#include <type_traits>

#include "device_utils.h"
#include "launch.h"

#ifndef LBC_QUANT_UNROLL
#define LBC_QUANT_UNROLL 4
#endif

namespace lbc {
namespace quant {


// torch type promotion for "a (op) b" restricted to {float, f16, bf16}.
template <typename A, typename B> struct promote { using type = float; };
template <typename A> struct promote<A, A> { using type = A; };
template <typename A> struct promote<A, void> { using type = A; };

template <typename T> struct or_float { using type = T; };
template <> struct or_float<void> { using type = float; };

// Stores of the interior blocks under the streaming mode, settled at the level of a pipeline, not of this kernel
// alone.  Without error feedback the codes are the only output and carry the non-temporal hint like the loads:
// plain or written-through code stores make the kernel 3-4 % faster when it is timed alone (26 M fp32 elements:
// 21.3 us written through, 21.4 plain, 21.9 non-temporal), but the lines they leave behind are paid for by the
// kernel that follows (a quantize -> shard-reduce step: 32.0 us non-temporal, 32.6 written through, 33.0 plain;
// the four-launch reduce-scatter plan 99.1 / 101.8 / 103.3 us).  With error feedback the residual is the large
// output and keeps the hint, and the codes are written through: a 613-bucket stream of (error-feedback quantize,
// shard reduce) measured 20.17 ms that way against 20.74 ms with both non-temporal, 20.75 both written through,
// 21.57 both plain and 21.97 the other way round; the 52 M-element bucket alone 89.9 against 93.2 us.
// That holds for chunks, which leave for other ranks.  The one payload of a whole tensor is read on this GPU next, by its
// decode or by a reduce that has it among its inputs: kStreamKept and kStreamThrough, chosen in quant_pack.hip's launch_tiles.
template <bool HAS_RESIDUAL, int MODE> constexpr int quant_code_store_policy() {
    if (MODE < kStream || MODE == kStreamKept) return kCached;
    return HAS_RESIDUAL || MODE == kStreamThrough ? kSc1Bit : kNtBit;
}

// Tiles in flight per wavefront for a tensor that keeps the chip busy for a while: four of four elements a lane, two of
// eight (a pure 16-bit call; four of eight fill 106 registers when a residual takes part, four wavefronts a SIMD: a 13.1 M
// bf16 bucket with a bf16 residual as eight chunks 20.9 us with two, 21.9 with four).
template <int VEC> constexpr int quant_unroll() { return VEC == 8 ? LBC_QUANT_UNROLL / 2 : LBC_QUANT_UNROLL; }

template <int VEC, int TILES> struct quant_tiling {
    static constexpr int TILE = kWave * VEC;        // elements per wavefront step
    static constexpr int UNROLL = TILES;            // tiles in flight per wavefront
    static constexpr int BLOCK_ELEMS = TILE * kWavesPerBlock * UNROLL;
};

// XT input, RT residual (void = none), DT type `restored` is rounded to.  Optional outputs besides the payload:
// `restored` (DT), `new_residual` = p - restored (promotion of p's type and DT) and `prepared` = p itself (p's type).
// One workgroup's share: block `block_x` of `grid_x` along the chunk, destination chunk `chunk`.
template <typename XT, typename RT, typename DT, int G, int VEC, int MODE, int TILES = quant_unroll<VEC>()>
__device__ __forceinline__ void quant_pack_block(const QuantArgs &a, unsigned block_x, unsigned grid_x, unsigned chunk_index) {
    using T = quant_tiling<VEC, TILES>;
    using PT = typename promote<XT, RT>::type;  // type of p = x + r
    using NT = typename promote<PT, DT>::type;  // type of p - restored
    using RLoad = typename or_float<RT>::type;  // placeholder when there is no residual
    constexpr bool HAS_R = !is_void_t<RT>::value;
    constexpr int LPG = G / VEC;                // lanes per group
    constexpr int UNROLL = T::UNROLL;
    static_assert(LPG >= 1 && LPG <= 16, "a group must fit one DPP row");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t chunk = chunk_index;
    const int64_t chunk_start = chunk * a.shard_numel;
    int64_t valid = a.numel - chunk_start;  // live elements of this chunk
    valid = valid < 0 ? 0 : (valid > a.shard_numel ? a.shard_numel : valid);
    const int64_t groups = (a.shard_numel + G - 1) / G;
    const int64_t padded = groups * G;

    const XT *__restrict__ x = static_cast<const XT *>(a.x) + chunk_start;
    const RLoad *r = HAS_R ? static_cast<const RLoad *>(a.residual) + chunk_start : nullptr;  // may alias new_r
    int8_t *__restrict__ codes = reinterpret_cast<int8_t *>(a.codes_base + chunk * a.payload_stride);
    float *__restrict__ scales = reinterpret_cast<float *>(a.scales_base + chunk * a.payload_stride);
    NT *new_r = a.new_residual ? static_cast<NT *>(a.new_residual) + chunk_start : nullptr;
    DT *__restrict__ restored = a.restored ? static_cast<DT *>(a.restored) + chunk_start : nullptr;
    PT *__restrict__ prepared = a.prepared ? static_cast<PT *>(a.prepared) + chunk_start : nullptr;

    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(block_x, grid_x, T::BLOCK_ELEMS)) * T::BLOCK_ELEMS;
    if (block_first >= padded) return;

    // One pass over the block's tiles, every load issued before the first use.  WHOLE: all of the block's elements are
    // live.  Whole blocks of aligned tensors address every stream through one descriptor over the block's span; the
    // rest (the block at a chunk's end, tensors at element alignment) goes through 64-bit addresses, with a lane's
    // vector cut short where the chunk ends.  The last block used to be walked element by element, a chain of up to
    // 4 * VEC dependent round trips to memory, and unaligned tensors were walked that way throughout: 9,830,417 bf16
    // elements as eight chunks (odd chunk starts) 20.0 us then, 8.0 us now (7.5 us aligned), 52,428,801 fp32 62.2 and
    // 41.1 us, with an fp32 residual (9.8 M bf16) 46.0 and 21.4 us; one 10,007-element tensor 2.9 and 2.4 us.  At
    // element alignment the non-temporal hint pays on the loads (8.0 against 8.9 us without) and not on the stores,
    // whose lines two wavefronts share (residual: 22.1 against 21.6 us).
    auto tiles = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        constexpr bool BUFFERS = WHOLE && MODE != kUnaligned;
        constexpr bool kLoadNt = MODE >= kStream || MODE == kUnaligned;
        constexpr bool kStoreNt = MODE >= kStream;
        constexpr int kLoad = policy_of<MODE>();
        // With several tiles a wavefront the outputs beside the codes leave with the non-temporal hint and written through, else with the
        // hint alone: the reduce that reads the sum next finds it nearer.  nt alone / both, GPU us with three states in rotation (and
        // beyond the last-level cache): local step of 52.4 M bf16 elements 105.9 / 101.4 (117.0 / 111.6), 26.2 M fp32 71.5 / 69.3, of one
        // tile a wavefront 2 M bf16 6.04 / 5.99 (6.35 / 6.63); the quantize that writes the sum, 24 M bf16 28.1 / 27.1 (27.9 / 26.9), 12 M fp32
        // 26.6 / 25.7 (26.4 / 25.5); with the reduce behind it, of one tile a wavefront, four fp32 payloads of 0.05 MiB 4.5 / 4.9 (5.1 / 5.4), 2 MiB
        // 6.5 / 7.0 (7.3 / 7.4), three bf16 of 1.6 MiB 6.9 / 7.3 (7.5 / 7.6), eight fp32 of 2.4 MiB 6.9 / 7.4 (7.7 / 8.0).
        constexpr int kSideStore = TILES > 1 && MODE >= kStream ? kNtBit | kSc1Bit : policy_of<MODE>();
        constexpr int kCodeStore = quant_code_store_policy<HAS_R, MODE>();
        XT xv[UNROLL][VEC];
        RLoad rv[UNROLL][VEC];
        uint32_t at[UNROLL];   // element offset inside the block
        const int64_t live_here = valid - block_first, padded_here = padded - block_first;
        const buffer_t x_b = buffer_over(x + block_first, T::BLOCK_ELEMS * sizeof(XT));
        const buffer_t r_b = buffer_over(HAS_R ? r + block_first : nullptr, T::BLOCK_ELEMS * sizeof(RLoad));
        // The order in which whole blocks issue the two tensors' loads is worth up to 3 % where a wavefront has four tiles, and
        // left alone the scheduler changes it with every change to the arithmetic behind: the residual's loads follow two
        // tiles behind the input's (x0 x1 x2 r0 x3 r1 r2 r3).  us of the local step, input first / tile by tile / residual
        // first tile by tile / residual first / this: 52.4 M bf16 elements 107.1 / 106.5 / 106.1 / 105.9 / 105.4, 26.2 M fp32
        // 73.3 / 70.9 / 71.2 / 71.3 / 70.9.
        constexpr int kLead = UNROLL > 2 ? 2 : 0;
        auto load_r = [&](int u) __attribute__((always_inline)) {
            buffer_load<RLoad, VEC, kLoad>(r_b, at[u] * sizeof(RLoad), rv[u]);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            at[u] = static_cast<uint32_t>(tile_in_block<UNROLL>(u, wave)) * T::TILE + lane * VEC;
            if constexpr (BUFFERS) {
                buffer_load<XT, VEC, kLoad>(x_b, at[u] * sizeof(XT), xv[u]);
                if constexpr (HAS_R) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (u >= kLead) load_r(u - kLead);
                }
            } else if constexpr (WHOLE) {
                load_any<XT, VEC, kLoadNt>(x + block_first + at[u], xv[u]);
                if constexpr (HAS_R) load_any<RLoad, VEC, kLoadNt>(r + block_first + at[u], rv[u]);
            } else {
                load_live<XT, VEC, kLoadNt>(x + block_first + at[u], live_here - at[u], xv[u]);
                if constexpr (HAS_R) load_live<RLoad, VEC, kLoadNt>(r + block_first + at[u], live_here - at[u], rv[u]);
            }
        }
        if constexpr (BUFFERS && HAS_R) {
#pragma unroll
            for (int u = UNROLL - kLead; u < UNROLL; ++u) load_r(u);
        }
        const buffer_t codes_b = buffer_over(codes + block_first, T::BLOCK_ELEMS);
        const buffer_t scales_b = buffer_over(scales + block_first / G, T::BLOCK_ELEMS / G * 4);
        // `out` of element type E, the block's part of the stream at `base`
        auto store_side = [&](auto *base, uint32_t offset, const auto &out) __attribute__((always_inline)) {
            using E = typename std::remove_pointer<decltype(base)>::type;
            if constexpr (BUFFERS) buffer_store<E, VEC, kSideStore>(buffer_over(base + block_first, T::BLOCK_ELEMS * sizeof(E)), offset * sizeof(E), out);
            else if constexpr (WHOLE) store_any<E, VEC, kStoreNt>(base + block_first + offset, out);
            else store_live<E, VEC, kStoreNt>(base + block_first + offset, live_here - offset, out);
        };
        float p[UNROLL][VEC];
        uint32_t absmax[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                p[u][i] = widen(xv[u][i]);
                if constexpr (HAS_R) p[u][i] += widen(rv[u][i]);
            }
            if constexpr (HAS_R) round_through_all<PT, VEC>(p[u]);
            // every lane of a row takes part; elements past the end count as zeros
            absmax[u] = group_absmax_bits<VEC, LPG>(p[u]);
        }
        // The scale of a group and its reciprocal cost ~10 instructions, and after the butterflies every lane of a
        // group holds the maxima of all four tiles.  With four tiles and at least four lanes per group the lanes of
        // a quad split the work: lane j of the quad takes tile j, and quad broadcasts hand the four results round.
        // Same operations on the same values as one computation per tile; some 20 instructions fewer per wavefront.
        constexpr bool kSplit = UNROLL == 4 && LPG >= 4;
        float scale[UNROLL], recip[UNROLL];
        auto store_scale = [&](uint32_t element, float value) __attribute__((always_inline)) {
            const float one[1] = {value};
            if constexpr (BUFFERS) buffer_store<float, 1, kCached>(scales_b, element / G * 4, one);
            else if (WHOLE || element < padded_here) scales[(block_first + element) / G] = value;
        };
        if constexpr (kSplit) {
            const int j = lane & 3;
            const uint32_t low = (j & 1) ? absmax[1] : absmax[0], high = (j & 1) ? absmax[3] : absmax[2];
            const float mine = scale_from_absmax(as_f32((j & 2) ? high : low));
            const float mine_recip = reciprocal_of_scale(mine);
            scale[0] = quad_broadcast<0>(mine); recip[0] = quad_broadcast<0>(mine_recip);
            scale[1] = quad_broadcast<1>(mine); recip[1] = quad_broadcast<1>(mine_recip);
            scale[2] = quad_broadcast<2>(mine); recip[2] = quad_broadcast<2>(mine_recip);
            scale[3] = quad_broadcast<3>(mine); recip[3] = quad_broadcast<3>(mine_recip);
            if ((lane & (LPG - 1)) < 4)     // the first quad of every group writes the four scales in one store
                store_scale(static_cast<uint32_t>(tile_in_block<UNROLL>(j, wave)) * T::TILE + lane * VEC, mine);
        } else {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                scale[u] = scale_from_absmax(as_f32(absmax[u]));
                recip[u] = reciprocal_of_scale(scale[u]);
                if ((lane & (LPG - 1)) == 0) store_scale(at[u], scale[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            int c[VEC];
            const bool no_codes = scale_not_finite(scale[u]);     // then every code of the group is 0
            encode_group_finite<VEC>(p[u], scale[u], recip[u], c);

            uint32_t words[VEC / 4];
#pragma unroll
            for (int k = 0; k < VEC / 4; ++k) {                   // one select per packed word, not per code
                const uint32_t word = pack4(c[4 * k], c[4 * k + 1], c[4 * k + 2], c[4 * k + 3]);
                words[k] = no_codes ? 0u : word;
            }
            if constexpr (BUFFERS) {
                buffer_store<uint32_t, VEC / 4, kCodeStore>(codes_b, at[u], words);
            } else if (WHOLE || at[u] < padded_here) {            // a lane's codes lie inside the padded range together
                constexpr int kCodeAlign = MODE == kUnaligned ? 1 : VEC;
                store_any<uint32_t, VEC / 4, false, kCodeAlign>(reinterpret_cast<uint32_t *>(codes + block_first + at[u]), words);
            }

            if (prepared != nullptr) {
                PT prep_out[VEC];
                narrow_all<PT, VEC>(p[u], prep_out);
                store_side(prepared, at[u], prep_out);
            }
            if (new_r != nullptr || restored != nullptr) {
                float rest[VEC], diff[VEC];
                DT rest_out[VEC];
                NT diff_out[VEC];
#pragma unroll
                for (int i = 0; i < VEC; ++i) rest[i] = (no_codes ? 0.0f : code_value(c[i])) * scale[u];
                round_through_all<DT, VEC>(rest);
#pragma unroll
                for (int i = 0; i < VEC; ++i) diff[i] = p[u][i] - rest[i];
                narrow_all<DT, VEC>(rest, rest_out);
                narrow_all<NT, VEC>(diff, diff_out);
                if (restored != nullptr) store_side(restored, at[u], rest_out);
                if (new_r != nullptr) store_side(new_r, at[u], diff_out);
            }
        }
    };
    if (block_first + T::BLOCK_ELEMS <= valid) tiles(std::true_type{});
    else tiles(std::false_type{});
}

}  // namespace quant
}  // namespace lbc
