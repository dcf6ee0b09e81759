// Device side of the decode-side kernels (fused dequant-reduce, reduce + requantize, decode of shard payloads):
// what one workgroup does.  Shared by the kernels of their own and by the kernels that carry several stages of a
// bucket stream in one grid.
#pragma once

#include <type_traits>

#include "device_utils.h"
#include "launch.h"

namespace lbc {
namespace reduce {


#ifndef LBC_DECODE_UNROLL
#define LBC_DECODE_UNROLL 1
#endif
// W payloads give 2*W loads per tile; with one or two payloads a second tile in
// flight per wavefront is needed to cover the memory latency.
template <typename OT, int W = 8> struct decode_tiling {
    static constexpr int VEC = sizeof(OT) == 4 ? 4 : 8;
    static constexpr int TILE = kWave * VEC;
    static constexpr int UNROLL = W <= 2 ? 2 * LBC_DECODE_UNROLL : LBC_DECODE_UNROLL;
    static constexpr int BLOCK_ELEMS = TILE * kWavesPerBlock * UNROLL;
};

// Cache policy of the code loads in streaming mode, from measurement on 100 MiB buckets: with one to
// three payloads the output dominates the traffic and cacheable code loads are ~13 % faster; from
// four payloads on the codes dominate and the non-temporal hint wins by ~9 %.
template <int W> __device__ __forceinline__ constexpr int code_load_mode(int mode) {
    return mode == kStream && W < 4 ? kVector : mode;
}
// Cache policy of the fused reduce under the streaming modes, from sweeps of every load/store policy pair at
// W = 1, 2, 4, 8 on 3.3 M, 6.6 M and 26 M fp32 elements with buffers rotating through 650 MB.  The non-temporal
// hint pays on the direction that carries most of the bytes and costs when both directions carry it:
//   reads/writes < 0.8  (W = 1, 2 for fp32)  plain code loads, non-temporal stores       (26 M, W = 1: 19.0 us; with
//                                             non-temporal loads as well 24.8 us)
//   up to 1.6           (W = 4; for 16-bit    non-temporal loads; stores non-temporal (two 16-bit payloads: written
//                        outputs W = 2)       through beside the hint unless the sum is loaded early), or written
//                                             through without it for outputs beyond the L2s
//   above               (W = 8)               non-temporal loads; plain stores while the output fits the L2s
//                                             (3.3 M: 7.9 us against 8.1 written through, 8.4 non-temporal - the
//                                             write-back then overlaps the next kernel's ramp), written through
//                                             beyond (26 M: 47.3 us against 50.2 plain, 53.6 non-temporal)
// The host picks kStream or kStreamThrough by the size of the output.  The choice holds inside a pipeline as well:
// a quantize -> shard-reduce step measured 31.7 us with these stores against 32.2-32.5 us with any other pair, and
// a 613-bucket stream of (error-feedback quantize, shard reduce) 20.69 ms against 20.8-21.2 ms.
template <typename OT, int W> constexpr int read_write_class() {
    constexpr int reads16 = W * 17, writes16 = static_cast<int>(sizeof(OT)) * 16;   // bytes per element, x16
    return reads16 * 10 < writes16 * 8 ? 0 : (reads16 * 10 < writes16 * 16 ? 1 : 2);
}
template <typename OT, int W, int MODE> constexpr int code_policy() {
    return MODE >= kStream && read_write_class<OT, W>() >= 1 ? kNtBit : kCached;
}
template <typename OT, int W, int MODE, bool EARLY_SUM> constexpr int reduce_store_policy() {
    if (MODE < kStream) return kCached;
    if (read_write_class<OT, W>() == 0) return kNtBit;
    if (MODE == kStreamThrough) return kSc1Bit;
    return read_write_class<OT, W>() == 1 ? (W <= 2 && !EARLY_SUM ? kNtBit | kSc1Bit : kNtBit) : kCached;
}

// Whether a call with error feedback has a kernel whose whole blocks issue the load of `prepared` together with the codes', and takes
// it for an output of `bytes`; else they load it behind the outputs' stores.  Early it is one round trip to memory less.  A kernel of its
// own, because the load and its branch cost calls without feedback 3 to 8 % of the reduce (eight bf16 payloads 23,552 elements 2.6 ->
// 2.8 us, 0.7 M 3.4 -> 3.6).  GPU us of the all_gather hook's two launches, late / early, three states in rotation (and beyond the last-level
// cache): one payload fp32 1.5 MiB 6.7 / 5.8 (7.0 / 6.1), two of fp32 2 MiB 6.8 / 5.9 (7.3 / 6.5), 50 MiB 60.9 / 58.1 (60.7 / 58.3), eight of bf16 0.5 MiB
// 5.8 / 5.4 (6.8 / 6.1), 3 MiB 11.1 / 9.9 (12.0 / 10.8), 20 MiB 38.7 / 37.9 (42.4 / 41.7).  Where reads and writes are about even (class 1) only two
// payloads, up to where the outputs are written through: two of bf16 2.5 MiB 8.3 / 7.4 (8.7 / 7.8), 5 MiB 11.0 / 10.2 (11.2 / 10.9), 10 MiB 17.4 / 17.5
// (17.5 / 17.6); four of fp32 8 MiB 13.5 / 14.4.  Three fp32 payloads gain to 6 MiB (11.0 / 10.5 (11.6 / 11.2)) and from 24 MiB on, between them
// they lose (11 MiB 17.5 / 18.3 (18.0 / 18.6)).
template <typename OT, int W, int MODE> constexpr bool prepared_early() {
    return MODE >= kStream && (read_write_class<OT, W>() != 1 || (W <= 2 && MODE != kStreamThrough));
}
template <typename OT, int W, int MODE> bool takes_early(int64_t bytes) {
    return !(sizeof(OT) == 4 && W == 3 && MODE == kStream && bytes >= int64_t{13} << 19);
}

// The VEC codes of a lane, from any address under kUnaligned.
template <int VEC, int MODE>
__device__ __forceinline__ void load_codes(const int8_t *__restrict__ p, uint32_t (&w)[VEC / 4]) {
    load_any<uint32_t, VEC / 4, MODE == kStream, MODE == kUnaligned ? 1 : VEC>(reinterpret_cast<const uint32_t *>(p), w);
}

// ---------------------------------------------------------------------------
// fused dequant-reduce
// ---------------------------------------------------------------------------
// One workgroup's share: block `block_x` of a grid of `grid_x` workgroups.  EARLY_SUM: the call has error feedback, and whole blocks load
// `prepared` with the codes.
template <typename OT, int G, int W, int MODE, bool EARLY_SUM = false>
__device__ __forceinline__ void dequant_reduce_block(const ReduceArgs &a, unsigned block_x, unsigned grid_x) {
    using T = decode_tiling<OT, W>;
    constexpr int VEC = T::VEC;
    constexpr int UNROLL = T::UNROLL;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    // every XCD walks one contiguous eighth of the shard at any size: with the policies above that measured
    // 6-15 % faster than the round-robin order from 3 M to 26 M elements (W = 8), and no slower at W = 1, 2, 4
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block<true>(block_x, grid_x, T::BLOCK_ELEMS)) * T::BLOCK_ELEMS;
    OT *__restrict__ out = static_cast<OT *>(a.out);
    const OT *prepared = static_cast<const OT *>(a.prepared);  // may alias new_r
    OT *new_r = static_cast<OT *>(a.new_residual);
    const bool mean = a.divisor != 1.0f;

    // One pass over the block's tiles with the codes and scales of all of them issued before the arithmetic (`prepared`
    // with them in the last block; in whole blocks under EARLY_SUM, else tile by tile after the tile's outputs).  WHOLE:
    // all of the block's outputs exist.  Whole blocks of aligned tensors use one descriptor per stream over the block's span and 32-bit offsets
    // per lane; the block at the end and tensors at element alignment use 64-bit addresses, a lane's vector cut short
    // at the end.  (A payload holds whole groups, so a lane with one live output may read all of its codes.)  Walked
    // element by element, that last block was the longest chain of the kernel: 3,186,579 bf16 outputs of two payloads
    // with error feedback 11.0 us, now 6.6 us, as long as whole blocks take; 1,228,803 fp32 outputs of eight payloads at
    // an odd start 10.9 and 4.5 us.
    auto tiles = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        constexpr bool BUFFERS = WHOLE && MODE != kUnaligned;
        constexpr int kLike = MODE == kUnaligned ? static_cast<int>(kStream) : MODE;   // policies as in the streaming mode
        constexpr int kCodes = code_policy<OT, W, kLike>();
        constexpr int kLoad = policy_of<kLike>();
        constexpr int kStore = reduce_store_policy<OT, W, kLike, EARLY_SUM>();
        // What the stores without a descriptor take of it.  Two bf16 payloads at an odd output, plain / non-temporal, beyond the
        // last-level cache: with feedback 1 M elements 4.73 / 4.69 us, 8 M 14.9 / 14.5, 13.1 M 22.4 / 22.4, without it 8 M 8.2 / 7.8,
        // 26.2 M 21.0 / 19.9.  (Three tensors in rotation, with feedback: 3.2 M 7.1 / 6.6, 13.1 M 19.3 / 22.0.)
        constexpr bool kStoreNt = (kStore & kNtBit) != 0;
        constexpr int kCodeAlign = MODE == kUnaligned ? 1 : VEC;
        constexpr bool kEarly = BUFFERS && EARLY_SUM;
        uint32_t words[UNROLL][W][VEC / 4];
        float scale[UNROLL][W];
        OT pv[UNROLL][VEC];
        uint32_t at[UNROLL];   // element offset inside the block
        const int64_t live_here = a.numel - block_first;
        const buffer_t prepared_b = buffer_over(prepared + block_first, T::BLOCK_ELEMS * sizeof(OT));
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) at[u] = static_cast<uint32_t>(tile_in_block<UNROLL>(u, wave)) * T::TILE + lane * VEC;
#pragma unroll
        for (int r = 0; r < W; ++r) {
            const buffer_t codes = buffer_over(a.codes[r] + block_first, T::BLOCK_ELEMS);
            const buffer_t scales = buffer_over(a.scales[r] + block_first / G, T::BLOCK_ELEMS / G * 4);
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                if constexpr (BUFFERS) {
                    buffer_load<uint32_t, VEC / 4, kCodes>(codes, at[u], words[u][r]);
                    float one[1];
                    buffer_load<float, 1, kCached>(scales, at[u] / G * 4, one);
                    scale[u][r] = one[0];
                } else {
#pragma unroll
                    for (int k = 0; k < VEC / 4; ++k) words[u][r][k] = 0;
                    scale[u][r] = 0.0f;
                    if (WHOLE || at[u] < live_here) {
                        load_any<uint32_t, VEC / 4, kCodes == kNtBit, kCodeAlign>(
                            reinterpret_cast<const uint32_t *>(a.codes[r] + block_first + at[u]), words[u][r]);
                        scale[u][r] = a.scales[r][(block_first + at[u]) / G];
                    }
                }
            }
        }
        if constexpr (kEarly) {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) buffer_load<OT, VEC, kLoad>(prepared_b, at[u] * sizeof(OT), pv[u]);
        } else if (!WHOLE && (EARLY_SUM || new_r != nullptr)) {   // the end of the tensor: nothing else hides this load
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) load_live<OT, VEC, kLoad == kNtBit>(prepared + block_first + at[u], live_here - at[u], pv[u]);
        }
        const buffer_t out_b = buffer_over(out + block_first, T::BLOCK_ELEMS * sizeof(OT));
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            float acc[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = code_to_float(words[u][0][i / 4], i % 4) * scale[u][0];
            round_through_all<OT, VEC>(acc);
#pragma unroll
            for (int r = 1; r < W; ++r) {
                float t[VEC];
#pragma unroll
                for (int i = 0; i < VEC; ++i) t[i] = code_to_float(words[u][r][i / 4], i % 4) * scale[u][r];
                round_through_all<OT, VEC>(t);
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc[i] += t[i];
                round_through_all<OT, VEC>(acc);
            }
            if (mean) divide_all<OT, VEC>(acc, a.divisor);
            OT o[VEC];
            narrow_all<OT, VEC>(acc, o);
            if constexpr (BUFFERS) buffer_store<OT, VEC, kStore>(out_b, at[u] * sizeof(OT), o);
            else if constexpr (WHOLE) store_any<OT, VEC, kStoreNt>(out + block_first + at[u], o);
            else store_live<OT, VEC, kStoreNt>(out + block_first + at[u], live_here - at[u], o);
            if (EARLY_SUM || new_r != nullptr) {
                OT d[VEC];
                if constexpr (BUFFERS && !kEarly) buffer_load<OT, VEC, kLoad>(prepared_b, at[u] * sizeof(OT), pv[u]);
                else if constexpr (WHOLE && !BUFFERS) load_any<OT, VEC, kLoad == kNtBit>(prepared + block_first + at[u], pv[u]);
#pragma unroll
                for (int i = 0; i < VEC; ++i) d[i] = narrow<OT>(widen(pv[u][i]) - acc[i]);
                if constexpr (BUFFERS) buffer_store<OT, VEC, kStore>(buffer_over(new_r + block_first, T::BLOCK_ELEMS * sizeof(OT)), at[u] * sizeof(OT), d);
                else if constexpr (WHOLE) store_any<OT, VEC, kStoreNt>(new_r + block_first + at[u], d);
                else store_live<OT, VEC, kStoreNt>(new_r + block_first + at[u], live_here - at[u], d);
            }
        }
    };
    if (block_first + T::BLOCK_ELEMS <= a.numel) tiles(std::true_type{});
    else tiles(std::false_type{});
}

// ---------------------------------------------------------------------------
// fused dequant-reduce + requantize (reduce-scatter shard -> all-gather payload)
// ---------------------------------------------------------------------------
// The reduced shard never reaches memory: each lane folds its 4 elements over the W payloads exactly as
// dequant_reduce_kernel does for an output of type MT (every partial sum rounded to MT, true division for
// the mean), the group maximum is taken across the lanes of the group and the codes and the scale of the
// new payload are written.  Elements past numel count as zeros, as the zero padding of a separate
// quantize would.  Reads W*(g+4)/g bytes and writes (g+4)/g bytes per element.
// Elements per lane of the fused reduce + requantize: 4 (one dword of codes per payload, 16 lanes per group
// of 64) measured 3-4 % faster on a full bucket than 8 and the same on shards.
constexpr int kReduceQuantVec = 4;
constexpr int kReduceQuantBlockElems = kWave * kReduceQuantVec * kWavesPerBlock;

// One workgroup's share: block `block_x` of a grid of `grid_x` workgroups.  W payloads; 0: as many as the call says, the
// absent ones skipped by uniform branches.
template <typename MT, int G, int W, int MODE>
__device__ __forceinline__ void dequant_reduce_quant_block(const ReduceQuantArgs &a, unsigned block_x, unsigned grid_x) {
    constexpr int VEC = kReduceQuantVec;
    constexpr int MAX = W == 0 ? kMaxPayloads : W;
    const int world = W == 0 ? a.world : W;
    constexpr int LPG = G / VEC;
    constexpr int TILE = kWave * VEC;
    constexpr int BLOCK_ELEMS = TILE * kWavesPerBlock;
    static_assert(LPG >= 1 && LPG <= 16, "a group must fit one DPP row");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t padded = (a.numel + G - 1) / G * G;
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block<true>(block_x, grid_x, BLOCK_ELEMS)) * BLOCK_ELEMS;
    const uint32_t at = static_cast<uint32_t>(wave) * TILE + lane * VEC;   // element offset inside the block
    const int64_t e0 = block_first + at;
    const bool live = e0 < padded;     // whole lanes: padded and e0 are multiples of VEC
    const bool mean = a.divisor != 1.0f;

    float p[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) p[i] = 0.0f;
    if (live) {
        uint32_t words[MAX][VEC / 4];
        float scale[MAX];
        const int64_t g = e0 / G;
#pragma unroll
        for (int r = 0; r < MAX; ++r) {
            if (r >= world) break;
            // Two loads a payload: with a descriptor for each and one offset for all, no 64-bit address is formed per lane (the plan's
            // three launches on 26.2 M bf16 elements of eight ranks 35.5 -> 34.9 us, on 9.8 M 17.55 -> 17.4).
            if constexpr (MODE != kUnaligned) {
                buffer_load<uint32_t, VEC / 4, policy_of<code_load_mode<MAX>(MODE)>()>(buffer_over(a.codes[r] + block_first, BLOCK_ELEMS), at, words[r]);
                float one[1];
                buffer_load<float, 1, kCached>(buffer_over(a.scales[r] + block_first / G, BLOCK_ELEMS / G * 4), at / G * 4, one);
                scale[r] = one[0];
            } else {
                load_codes<VEC, code_load_mode<MAX>(MODE)>(a.codes[r] + e0, words[r]);
                scale[r] = a.scales[r][g];
            }
        }
#pragma unroll
        for (int i = 0; i < VEC; ++i) p[i] = code_to_float(words[0][i / 4], i % 4) * scale[0];
        round_through_all<MT, VEC>(p);
#pragma unroll
        for (int r = 1; r < MAX; ++r) {
            if (r >= world) break;
            float t[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) t[i] = code_to_float(words[r][i / 4], i % 4) * scale[r];
            round_through_all<MT, VEC>(t);
#pragma unroll
            for (int i = 0; i < VEC; ++i) p[i] += t[i];
            round_through_all<MT, VEC>(p);
        }
        if (mean) divide_all<MT, VEC>(p, a.divisor);
        if (e0 + VEC > a.numel) {
#pragma unroll
            for (int i = 0; i < VEC; ++i) p[i] = e0 + i < a.numel ? p[i] : 0.0f;
        }
    }
    // every lane of the row takes part in the butterfly; lanes past the end contribute zeros
    const float out_scale = group_scale<VEC, LPG>(p);
    if (!live) return;
    int c[VEC];
    encode_group<VEC>(p, out_scale, c);
    uint32_t out_words[VEC / 4];
#pragma unroll
    for (int k = 0; k < VEC / 4; ++k) out_words[k] = pack4(c[4 * k], c[4 * k + 1], c[4 * k + 2], c[4 * k + 3]);
    store_any<uint32_t, VEC / 4, false, MODE == kUnaligned ? 1 : VEC>(reinterpret_cast<uint32_t *>(a.out_codes + e0), out_words);
    if ((lane & (LPG - 1)) == 0) a.out_scales[e0 / G] = out_scale;
}

// ---------------------------------------------------------------------------
// decode of one payload, or of `world` shard payloads into consecutive shards
// ---------------------------------------------------------------------------
template <int OP> __device__ __forceinline__ float combine(float old, float v) {
    if constexpr (OP == 1) return old + v;
    else if constexpr (OP == 2) return old > v ? old : v;
    else if constexpr (OP == 3) return old < v ? old : v;
    else return v;
}

#ifndef LBC_DECODE1_UNROLL
#define LBC_DECODE1_UNROLL 2
#endif
template <typename OT> struct decode1_tiling {
    static constexpr int VEC = decode_tiling<OT>::VEC;
    static constexpr int TILE = kWave * VEC;
    static constexpr int UNROLL = LBC_DECODE1_UNROLL;   // a single payload has few loads per tile: keep more tiles in flight
    static constexpr int BLOCK_ELEMS = TILE * kWavesPerBlock * UNROLL;
};

// One workgroup's share: block `block_x` of `grid_x` along shard `chunk_index`.  STREAM_STORE: cache policy of whole blocks of
// aligned outputs in the streaming mode.
template <typename OT, int G, int OP, int MODE, int STREAM_STORE = kNtBit>
__device__ __forceinline__ void decode_block(const DecodeArgs &a, unsigned block_x, unsigned grid_x, unsigned chunk_index) {
    using T = decode1_tiling<OT>;
    constexpr int VEC = T::VEC;
    constexpr int UNROLL = T::UNROLL;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int64_t chunk = chunk_index;
    const int64_t chunk_start = chunk * a.shard_numel;
    int64_t valid = a.total_numel - chunk_start;
    valid = valid < 0 ? 0 : (valid > a.shard_numel ? a.shard_numel : valid);
    const int8_t *__restrict__ codes = reinterpret_cast<const int8_t *>(a.codes_base + chunk * a.payload_stride);
    const float *__restrict__ scales = reinterpret_cast<const float *>(a.scales_base + chunk * a.payload_stride);
    OT *__restrict__ out = static_cast<OT *>(a.out) + chunk_start;
    const int64_t block_first = static_cast<int64_t>(xcd_contiguous_block(block_x, grid_x, T::BLOCK_ELEMS)) * T::BLOCK_ELEMS;
    if (block_first >= valid) return;

    // WHOLE: all of the block's outputs exist; otherwise a lane's vector is cut short at the end of the shard.  The codes and
    // scales of all tiles are issued first; what a combining decode adds to is loaded with them in the last block, and tile
    // by tile in whole ones.  At
    // element alignment the stores keep the non-temporal hint (52.4 M fp32 outputs in eight odd shards: 44.8 us with it,
    // 48.7 us without, 112.7 us element by element; 9.8 M bf16 6.4, 8.9 and 23.2 us).  A 100,001-element tensor whose
    // last block walked its elements one dependent load at a time took 4.1 us, now 2.0 us.
    auto tiles = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        constexpr bool kLoadNt = MODE == kStream || MODE == kUnaligned;
        constexpr int kAlign = MODE == kUnaligned ? sizeof(OT) : VEC * sizeof(OT);
        constexpr int kStore = MODE == kStream ? STREAM_STORE : kCached;
        const buffer_t out_b = buffer_over(out + block_first, T::BLOCK_ELEMS * sizeof(OT));
        uint32_t words[UNROLL][VEC / 4];
        float scale[UNROLL];
        OT o[UNROLL][VEC];
        int64_t e0[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            e0[u] = block_first + static_cast<int64_t>(tile_in_block<UNROLL>(u, wave)) * T::TILE + lane * VEC;
#pragma unroll
            for (int k = 0; k < VEC / 4; ++k) words[u][k] = 0;
            scale[u] = 0.0f;
            if (WHOLE || e0[u] < valid) {
                load_codes<VEC, code_load_mode<1>(MODE)>(codes + e0[u], words[u]);
                scale[u] = scales[e0[u] / G];
            }
            if constexpr (OP != 0 && !WHOLE) load_live<OT, VEC, kLoadNt>(out + e0[u], valid - e0[u], o[u]);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            if constexpr (OP != 0 && WHOLE) load_any<OT, VEC, kLoadNt, kAlign>(out + e0[u], o[u]);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                float v = round_through<OT>(code_to_float(words[u][i / 4], i % 4) * scale[u]);
                if constexpr (OP != 0) v = round_through<OT>(combine<OP>(widen(o[u][i]), v));
                o[u][i] = narrow<OT>(v);
            }
            if constexpr (WHOLE && MODE != kUnaligned) buffer_store<OT, VEC, kStore>(out_b, static_cast<uint32_t>(e0[u] - block_first) * sizeof(OT), o[u]);
            else if constexpr (WHOLE) store_any<OT, VEC, kLoadNt>(out + e0[u], o[u]);
            else store_live<OT, VEC, kLoadNt>(out + e0[u], valid - e0[u], o[u]);
        }
    };
    if (block_first + T::BLOCK_ELEMS <= valid) tiles(std::true_type{});
    else tiles(std::false_type{});
}

}  // namespace reduce
}  // namespace lbc
