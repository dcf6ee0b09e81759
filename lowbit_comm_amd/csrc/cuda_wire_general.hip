// The policies of the reference's CUDA extension beyond plain linear codes, in its payload format:
// non-linear 4-bit code books, stochastic rounding, the top-k side channel and the group maximum that
// a NaN resets (ccdl_comm/csrc/quantization/quant_kernel_fp32.cuh, quant_kernel.cuh, inner.cuh,
// dequant_kernel_fp32.cuh, dequant_kernel.cuh).  ccdl_cuda_ops.quantize / dequantize run these
// kernels for every policy; inputs are whole groups (gen_code_quant.py:164).
//
// Payload of a group, in words of the tensor's item size (quant_kernel_fp32.cuh:283-331,390-417):
//   [code words][scale]                                   top-k 0
//   [code words][scale][index][top1]                      top-k 1
//   [code words][scale][index1 | index2 << 8][top1][top2] top-k 2
// with the metadata behind each group's codes (compact) or behind all codes.  The top-k elements are
// stored as they are, encoded as zero, and the scale is the next largest magnitude.
//
// The reference walks a group with one thread, element by element: fp32 groups from element 0,
// fp16/bf16 groups from element 4 * ((group & 31) / (32 / (G / 4))) with wrap-around.  That order
// decides (a) which elements a NaN hides from the running maximum `(m > a) ? m : a`, (b) ties of the
// top-k search (fp32 compares with >=: the later element wins and zeros qualify; 16-bit compares
// with >: the earlier element of the scan wins and zeros do not), (c) which draw of the group's
// Philox stream an element receives.  Here a group lies across G/VEC lanes of a DPP row as in the
// other kernels, and each of the three is restated in an order-free form: (a) the maximum over the
// scan positions behind the last NaN, (b) the three largest keys (magnitude bits, tie-break rank),
// merged across the row, (c) Philox in counter mode - draw j of group s is word (offset + j) % 4
// of block (offset + j) / 4 of subsequence s, so a lane computes the blocks of its own elements.
#include "code_book_cells.h"
#include "device_utils.h"
#include "launch.h"
#include "wire_common.h"

namespace lbc {
namespace {

// inner.cuh:9-35, and the one-lookup form of the encoder built from them at compile time
__constant__ book_cells::Books kCodeBooks = book_cells::kBookSet;
__constant__ book_cells::Places kBookPlaces = book_cells::kPlaces, kBookFloors = book_cells::kFloors;
__constant__ book_cells::Gaps kBookGaps = book_cells::kGaps;

// Philox4x32-10: one block of four 32-bit words.  A round is two 32x32->64 multiplies and two three-way
// exclusive-ors; gfx950 has the latter as one instruction (v_bitop3_b32 with the truth table 0x96), which the
// compiler does not choose by itself for `a ^ b ^ c`.
__device__ __forceinline__ uint32_t xor3(uint32_t x, uint32_t y, uint32_t z) {
    return __builtin_amdgcn_bitop3_b32(x, y, z, 0x96);
}

__device__ __forceinline__ void philox_block(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1,
                                             uint32_t (&out)[4]) {
#pragma unroll
    for (int round = 0; round < 10; ++round) {
        if (round) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c0, p1 = static_cast<uint64_t>(0xCD9E8D57u) * c2;
        const uint32_t n0 = xor3(static_cast<uint32_t>(p1 >> 32), c1, k0), n2 = xor3(static_cast<uint32_t>(p0 >> 32), c3, k1);
        c0 = n0;
        c1 = static_cast<uint32_t>(p1);
        c2 = n2;
        c3 = static_cast<uint32_t>(p0);
    }
    out[0] = c0;
    out[1] = c1;
    out[2] = c2;
    out[3] = c3;
}

// Each wavefront keeps its own copy of the code book in LDS: written and read by the same wavefront, whose LDS
// operations execute in order, so no workgroup barrier stands between the first loads and the arithmetic.
__device__ __forceinline__ const float *wave_code_book(int kind, int lane) {
    __shared__ float books[kWavesPerBlock][16];
    float *book = books[threadIdx.x >> 6];
    if (kind != 0) {
        if (lane < 16) book[lane] = kCodeBooks.value[kind - 1][lane];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    return book;
}

// The workgroup's copy of a book's cell table (code_book_cells.h) in LDS, and for stochastic rounding (GAPS) of its entries
// with their gaps.  The loads are issued by `fetch`, ahead of the tensor's own, so that `publish` need not wait for those; every
// wavefront of the workgroup must come to `publish`, which ends in a workgroup barrier that orders LDS only.
template <bool GAPS> struct BlockCells {
    static constexpr int PER_THREAD = (book_cells::kCells + kBlock - 1) / kBlock;
    static_assert(sizeof(book_cells::Cell) == sizeof(u32x2) && alignof(book_cells::Cell) >= alignof(u32x2) &&
                      sizeof(book_cells::Gap) == sizeof(u32x4) && alignof(book_cells::Gap) >= alignof(u32x4),
                  "the tables are copied in whole entries");
    u32x2 held[PER_THREAD];
    u32x4 held_gap;
    const book_cells::Cell *cells;
    const book_cells::Gap *gaps;

    __device__ __forceinline__ void fetch(int kind) {
        const u32x2 *table = reinterpret_cast<const u32x2 *>((GAPS ? kBookFloors : kBookPlaces).entry[kind - 1]);
#pragma unroll
        for (int k = 0; k < PER_THREAD; ++k) {
            const int place = k * kBlock + threadIdx.x;
            if (place < book_cells::kCells) held[k] = table[place];
        }
        if (GAPS && threadIdx.x < 16) held_gap = reinterpret_cast<const u32x4 *>(kBookGaps.entry[kind - 1])[threadIdx.x];
    }
    __device__ __forceinline__ void publish() {
        __shared__ u32x2 cell_table[book_cells::kCells];
        __shared__ u32x4 gap_table[GAPS ? 16 : 1];
#pragma unroll
        for (int k = 0; k < PER_THREAD; ++k) {
            const int place = k * kBlock + threadIdx.x;
            if (place < book_cells::kCells) cell_table[place] = held[k];
        }
        if (GAPS && threadIdx.x < 16) gap_table[threadIdx.x] = held_gap;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        cells = reinterpret_cast<const book_cells::Cell *>(cell_table);
        gaps = reinterpret_cast<const book_cells::Gap *>(gap_table);
    }
};

__device__ __forceinline__ int meta_words_of(int topk) { return topk == 0 ? 1 : topk + 2; }

// ---------------------------------------------------------------------------------------------
// quantize: a wavefront owns one tile of 64 * EL elements (64 lanes x 32 bytes of the tensor)
// ---------------------------------------------------------------------------------------------
// Elements per lane: 32 bytes of the tensor, twice what the other kernels of this format give a lane.  What a
// policy costs per group - addresses, the NaN rule of the running maximum, the outlier searches, the division behind
// the scale - is spread over twice the elements, and a group's reductions cross half the lanes.  These kernels are
// bound by instruction work and latency, not by memory, so that is what counts (26.2 M elements, 16 against 32 bytes a
// lane: see the measurements at launch_general_quant_g).
template <typename T> constexpr int general_quant_elems() { return 32 / static_cast<int>(sizeof(T)); }

// The EL 4-bit codes of one lane -> its 32-bit words.  Four codes make one 16-bit unit with the first code on top; a
// 16-bit tensor's word holds two units, low half first, an fp32 tensor's word holds elements 0-3 in its upper half.
template <typename T, int EL>
__device__ __forceinline__ void pack_nibbles(const int (&c)[EL], uint32_t (&words)[EL / 8]) {
#pragma unroll
    for (int k = 0; k < EL / 8; ++k) {
        uint32_t unit[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            unit[h] = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) unit[h] |= (static_cast<uint32_t>(c[8 * k + 4 * h + i]) & 0xFu) << (12 - 4 * i);
        }
        words[k] = sizeof(T) == 4 ? (unit[0] << 16) | unit[1] : unit[0] | (unit[1] << 16);
    }
}

__device__ __forceinline__ uint32_t umed3(uint32_t x, uint32_t y, uint32_t z) {
    uint32_t m;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(m) : "v"(x), "v"(y), "v"(z));
    return m;
}

// first >= second >= third are the three largest keys a lane knows (0 = none; nonzero keys are unique inside a
// group).  Afterwards every lane of the group's LANES adjacent lanes holds the three largest of the group.  With
// p, q = max, min of the two firsts, r, s = max, min of the seconds and t = max of the thirds, the union's first is
// p, its second max(q, r) and its third max(min(q, r), s, t).  row_half_mirror and row_mirror act as xor 4 / xor 8
// because the lanes they pair within a quad (half) already agree.
template <int CTRL> __device__ __forceinline__ void merge_top3_step(uint32_t &first, uint32_t &second, uint32_t &third) {
    auto partner = [](uint32_t v) {
        return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true));
    };
    const uint32_t f = partner(first), g = partner(second), h = partner(third);
    const uint32_t p = first > f ? first : f, q = first > f ? f : first;
    const uint32_t r = second > g ? second : g, s = second > g ? g : second;
    const uint32_t t = third > h ? third : h;
    const uint32_t low = q < r ? q : r;
    first = p;
    second = q > r ? q : r;
    third = low > s ? (low > t ? low : t) : (s > t ? s : t);
}

template <int LANES> __device__ __forceinline__ void merge_top3(uint32_t &first, uint32_t &second, uint32_t &third) {
    static_assert(LANES == 1 || LANES == 2 || LANES == 4 || LANES == 8 || LANES == 16, "row-sized groups only");
    if constexpr (LANES >= 2) merge_top3_step<0xB1>(first, second, third);    // quad_perm [1,0,3,2]
    if constexpr (LANES >= 4) merge_top3_step<0x4E>(first, second, third);    // quad_perm [2,3,0,1]
    if constexpr (LANES >= 8) merge_top3_step<0x141>(first, second, third);   // row_half_mirror
    if constexpr (LANES >= 16) merge_top3_step<0x140>(first, second, third);  // row_mirror
}

// FIXED names the policy, so that the code of the others is not part of the kernel: bit 0 "no outlier channel", bit 1 "round
// to nearest", bit 2 "linear codes" (else a code book), bit 3 "stochastic rounding".  13 and 12: linear codes rounded
// stochastically, without and with outliers; 9 and 8: a code book likewise; 6: linear codes rounded to nearest with
// outliers (without them lbc_wire_quant_pack serves the call); 3 and 2: a code book rounded to nearest, without and with.
// EL: elements per lane, a multiple of 8 that divides G; a wavefront owns one tile of 64 * EL elements.
// Codes leave in plain stores: with the non-temporal hint a launch alone is up to 6 % faster, and what reads the payload
// next pays for it (quantize and decode of 26.2 M elements with two outliers: fp32 44.9 plain against 52.0 us, bf16 28.6
// against 31.4).
template <typename T, int G, int BIT, int FIXED, int EL>
__global__ __launch_bounds__(kBlock) void wire_general_quant_kernel(const WireGeneralQuantArgs a) {
    const int topk = (FIXED & 1) ? 0 : a.topk;
    constexpr bool STOCHASTIC = (FIXED & 8) != 0;
    using W = wire<T, BIT>;
    using RB = raw_bits<T>;
    using Raw = typename RB::type;
    constexpr int VEC = EL, LPG = G / VEC, ITEM = sizeof(T), CB = G * BIT / 8, WORDS = EL * BIT / 32;
    constexpr bool WIDE = ITEM == 4;
    static_assert(EL % 8 == 0 && EL % W::VEC == 0 && G % EL == 0 && LPG <= 16, "a group lies in 1..16 lanes of one DPP row");

    const int lane = threadIdx.x & (kWave - 1);
    const int meta_bytes = meta_words_of(topk) * ITEM;
    const int64_t groups = a.numel / G;
    constexpr int TILE = kWave * EL;
    const int64_t tile_first = (static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6)) * TILE;
    const int64_t e0 = tile_first + lane * VEC;
    const bool live = e0 < a.numel;      // numel is a multiple of G: dead lanes form whole dead groups

    constexpr bool BOOK = (FIXED & 4) == 0, STOCHASTIC_BOOK = BOOK && (FIXED & 8) != 0;
    BlockCells<STOCHASTIC_BOOK> table;
    if constexpr (BOOK) table.fetch(a.kind);
    // All of the wavefront's elements are asked for before anything else, and kept as whole dwords: 16-bit elements taken
    // apart inside the branch would be waited for there, ahead of the tables and of the draws (26.2 M bf16 elements with
    // two outliers, rounded stochastically, 23.7 against 22.4 us, 3.3 M 6.4 against 5.4).
    constexpr int PARTS = EL / W::VEC, DWORDS = W::VEC * ITEM / 4;
    uint32_t held[PARTS][DWORDS];
#pragma unroll
    for (int part = 0; part < PARTS; ++part)
#pragma unroll
        for (int i = 0; i < DWORDS; ++i) held[part][i] = 0;
    if (live) {   // instruction-bound: a cache hint only costs
#pragma unroll
        for (int part = 0; part < PARTS; ++part)
            load_words<DWORDS, ITEM, kPlain>(reinterpret_cast<const uint8_t *>(static_cast<const Raw *>(a.x) + e0 + part * W::VEC), held[part]);
    }
    if constexpr (BOOK) table.publish();
    if (tile_first >= a.numel) return;   // wavefront-uniform, behind the workgroup's barrier

    const int64_t group = e0 / G;
    const int k0 = static_cast<int>(e0 - group * G);
    const int start = scan_start<T, G>(group);
    // The draws depend on the element's place only: they are computed while its value is still on its way.
    float uniform[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) uniform[i] = 0.0f;
    if constexpr (STOCHASTIC) {
        const uint32_t key0 = static_cast<uint32_t>(a.seed), key1 = static_cast<uint32_t>(a.seed >> 32);
        const uint32_t sub0 = static_cast<uint32_t>(group), sub1 = static_cast<uint32_t>(static_cast<uint64_t>(group) >> 32);
        const int phase = static_cast<int>(a.offset & 3);
        // curand_uniform, (0, 1]: x * 2^-32 + 2^-33.  The product is exact, so the fused form rounds as the two steps do.
        auto to_uniform = [](uint32_t x) { return __builtin_fmaf(static_cast<float>(x), 0x1p-32f, 0x1p-33f); };
        uint64_t block[VEC / 4];
#pragma unroll
        for (int q = 0; q < VEC / 4; ++q)
            block[q] = (a.offset + static_cast<uint64_t>((k0 + 4 * q - start) & (G - 1))) >> 2;   // positions are multiples of 4
        uint32_t lo[VEC / 4][4];
#pragma unroll
        for (int q = 0; q < VEC / 4; ++q)
            philox_block(static_cast<uint32_t>(block[q]), static_cast<uint32_t>(block[q] >> 32), sub0, sub1, key0, key1, lo[q]);
        if (phase == 0) {   // uniform; the offsets torch hands out are multiples of four: one block a quad
#pragma unroll
            for (int q = 0; q < VEC / 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) uniform[4 * q + e] = to_uniform(lo[q][e]);
        } else {            // a quad's draws lie across two blocks
#pragma unroll
            for (int q = 0; q < VEC / 4; ++q) {
                uint32_t hi[4];
                philox_block(static_cast<uint32_t>(block[q] + 1), static_cast<uint32_t>((block[q] + 1) >> 32), sub0, sub1,
                             key0, key1, hi);
                const uint32_t w[8] = {lo[q][0], lo[q][1], lo[q][2], lo[q][3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    uniform[4 * q + e] = to_uniform(phase == 1 ? w[e + 1] : (phase == 2 ? w[e + 2] : w[e + 3]));
            }
        }
    }

    Raw raw[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i)
        raw[i] = static_cast<Raw>(held[i / W::VEC][i % W::VEC * ITEM / 4] >> (ITEM == 2 && (i & 1) ? 16 : 0));
    float v[VEC];
    uint32_t mag[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
        v[i] = value_of<T>(raw[i]);
        mag[i] = raw[i] & RB::ABS;
    }

    uint8_t *group_codes = a.payload + (a.compact ? group * (CB + meta_bytes) : group * CB);
    uint8_t *group_meta = a.compact ? group_codes + CB : a.payload + groups * CB + group * meta_bytes;

    uint32_t scale_raw;
    Raw meta[4] = {0, 0, 0, 0};   // [scale][indices][top1][top2]
    bool any_nan = true;   // does the wavefront hold one?
    uint32_t outlier[2] = {~0u, ~0u};   // place among the lane's elements, beyond them when another lane's
    if constexpr ((FIXED & 1) != 0) {
        scale_raw = running_max_raw<T, G, VEC>(mag, k0, start, &any_nan);
    } else {
        // The three largest candidates of the group, a candidate's key being its magnitude and a tie-break rank
        // (1..G, unique inside a group; the larger rank wins).  The sign travels below the rank, so that what the search
        // finds is the element itself: fetched from the tensor once more, at the end of a wavefront's chain, the two
        // outliers of a group made the 16-bit kernel 14 % slower (26.2 M bf16 elements 19.5 against 17.1 us).
        uint32_t best_key[3] = {0, 0, 0}, best_rank[2] = {0, 0};              // magnitude + 1, rank
        uint32_t best_raw[2] = {0, 0};                                        // the element as stored
        if constexpr (WIDE) {
            // Three rounds of "largest remaining candidate": the group maximum of the magnitude keys, then, among
            // the elements that hold it, the maximum of the ranks.
            uint32_t key[VEC], rank[VEC], top = 0;
#pragma unroll
            for (int i = 0; i < VEC; ++i) top = mag[i] > top ? mag[i] : top;
            any_nan = __ballot(top > RB::INF) != 0;   // wavefront-uniform
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                rank[i] = __builtin_amdgcn_alignbit(static_cast<uint32_t>(k0 + i + 1), raw[i], 31);   // sign below it
                key[i] = mag[i] + 1;                                          // 0 stands for "none"
            }
            if (any_nan) {
#pragma unroll
                for (int i = 0; i < VEC; ++i) key[i] = mag[i] <= RB::INF ? key[i] : 0;
            }
#pragma unroll
            for (int round = 0; round < 3; ++round) {
                if (round == 2 && topk == 1) break;                         // uniform
                uint32_t m = 0;
#pragma unroll
                for (int i = 0; i < VEC; ++i) m = key[i] > m ? key[i] : m;
                m = group_max_bits<LPG>(m);
                best_key[round] = m;
                if (round == 2) break;
                uint32_t r = 0;
#pragma unroll
                for (int i = 0; i < VEC; ++i) r = (key[i] == m && rank[i] > r) ? rank[i] : r;
                r = group_max_bits<LPG>(r);
                r = m == 0 ? 0 : r;
                best_rank[round] = r >> 1;
                best_raw[round] = (m - 1) | (r << 31);
#pragma unroll
                for (int i = 0; i < VEC; ++i) key[i] = rank[i] == r ? 0 : key[i];   // taken (r = 0 matches nobody)
            }
        } else {
            // A 16-bit magnitude, its rank less one and its sign share one 32-bit key, unique inside the group: the
            // loaded dword rotated so that the magnitude lies on top and the sign at the bottom, the rest masked out
            // and the rank or-ed in, the quad's part and the constant part apart.  A lane keeps the three
            // largest of its own keys in order (three instructions an element), and the group's lanes merge their
            // triples over the DPP butterfly (eight instructions a step): no rounds over the elements.  Zeros are no
            // candidates: their keys are below 2^17, under every candidate's, and are dropped from the result.  NaNs are no candidates either and their keys are above every
            // candidate's: the first pass does not look for them, and when one tops any group of the wavefront
            // (rare) the pass is repeated with every element checked.  Scan positions do not wrap inside four
            // adjacent elements (a lane's first element and the scan's start are multiples of four).
            constexpr uint32_t kBelow = 1u << 17, kAbove = (RB::INF << 17) | 0x1FFFFu;
            uint32_t largest, runner_up, bronze;
            auto search = [&](const bool checked) __attribute__((always_inline)) {
                largest = runner_up = bronze = 0;
                const uint32_t p0 = static_cast<uint32_t>(k0 - start) & (G - 1);
#pragma unroll
                for (int q = 0; q < VEC / 4; ++q) {
                    const uint32_t rank0 = (G - 4) ^ ((p0 + 4 * q) & (G - 1));   // rank - 1 = G - 1 - scan position
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int i = 4 * q + j;
                        const uint32_t pair = static_cast<uint32_t>(raw[i & ~1]) | static_cast<uint32_t>(raw[i | 1]) << 16;
                        const uint32_t turned = __builtin_amdgcn_alignbit(pair, pair, (i & 1) ? 31 : 15);
                        uint32_t key = (turned & 0xFFFE0001u) | (rank0 << 1) | (2 * (3 - j));
                        if (checked) key = (key >> 17) - 1u < RB::INF ? key : 0;
                        bronze = umed3(runner_up, bronze, key);
                        runner_up = umed3(largest, runner_up, key);
                        largest = key > largest ? key : largest;
                    }
                }
                merge_top3<LPG>(largest, runner_up, bronze);
            };
            search(false);
            any_nan = __ballot(largest > kAbove) != 0;   // wavefront-uniform
            if (any_nan) search(true);
            largest = largest < kBelow ? 0 : largest;
            runner_up = runner_up < kBelow ? 0 : runner_up;
            bronze = bronze < kBelow ? 0 : bronze;
            const uint32_t found[3] = {largest, runner_up, bronze};
#pragma unroll
            for (int round = 0; round < 3; ++round) {
                best_key[round] = found[round] == 0 ? 0 : (found[round] >> 17) + 1;
                if (round < 2) {
                    best_rank[round] = found[round] == 0 ? 0 : ((found[round] & 0x1FFFFu) >> 1) + 1;
                    best_raw[round] = (found[round] >> 17) | (found[round] << 15);
                }
            }
        }
        auto index_of = [&](uint32_t r) {
            return WIDE ? static_cast<int>(r) - 1 : ((G - static_cast<int>(r)) + start) & (G - 1);
        };
        const bool none = best_key[0] == 0, second_missing = best_key[1] == 0;
        const int index1 = none ? 0 : index_of(best_rank[0]);
        int index2 = -1;
        if (topk == 1) {
            // nothing comparable: the reference falls back to element 1 (as stored for fp32, its magnitude otherwise)
            const uint32_t element1 = WIDE ? static_cast<uint32_t>(raw[1]) : raw[1] & RB::ABS;
            const uint32_t fallback = static_cast<uint32_t>(__shfl(static_cast<int>(element1), lane & ~(LPG - 1)));
            scale_raw = none ? fallback : (best_key[1] == 0 ? 0u : best_key[1] - 1);
        } else {
            const bool lonely = !none && best_key[1] == 0;
            index2 = none ? 1 : (lonely ? ((index1 + 1) & (G - 1)) : index_of(best_rank[1]));
            scale_raw = (none || lonely || best_key[2] == 0) ? 0u : best_key[2] - 1;
        }
        // Outliers encode as 0.  A code book needs the elements gone (they lie above the scale); linear codes, which a
        // zero element always turns into 0 (the noise stays within +-1/2, which rounds to 0), are cleared in the
        // packed words: five instructions a word instead of three an element.
        if constexpr (FIXED & 4) {
            outlier[0] = static_cast<uint32_t>(index1 - k0);
            outlier[1] = static_cast<uint32_t>(index2 - k0);
        } else {
#pragma unroll
            for (int i = 0; i < VEC; ++i)
                if (k0 + i == index1 || k0 + i == index2) v[i] = 0.0f;
        }
        meta[1] = static_cast<Raw>(topk == 1 ? index1 : (index1 | (index2 << 8)));
        meta[2] = static_cast<Raw>(best_raw[0]);
        meta[3] = static_cast<Raw>(best_raw[1]);
        if (live && k0 == 0 && (none || second_missing)) {   // rare: an index that the search did not give
            const Raw *members = static_cast<const Raw *>(a.x) + group * G;
            meta[2] = members[index1];
            if (topk == 2) meta[3] = members[index2];
        }
    }
    meta[0] = static_cast<Raw>(scale_raw);
    auto store_meta = [&]() __attribute__((always_inline)) {
        if (live && k0 == 0) {
            Raw *words = reinterpret_cast<Raw *>(group_meta);
            if (topk == 2) {
                store_elems<Raw, 4, kPlain>(words, meta);
            } else if (topk == 1) {
                const Raw pair[2] = {meta[0], meta[1]};
                store_elems<Raw, 2, kPlain>(words, pair);
                words[2] = meta[2];
            } else {
                words[0] = meta[0];
            }
        }
    };

    float scale = value_of<T>(scale_raw);
    scale = scale < 1.0e-6f ? 1.0e-6f : scale;   // a NaN scale stays NaN and encodes every element as 0

    if constexpr (BOOK) {
        // A code book.  Rounded to nearest, the cell lookup answers v / scale without forming
        // the quotient: per element a fused multiply-add and an address, one LDS read, and four operations that leave
        // the comparison with the step in a sign bit and push it and the cell's code into a word of eight.  It
        // holds for a scale within 2^60 of 1 either way and |v| <= scale; the scale is at least 1e-6 here, and beside
        // outliers or a NaN an element may lie above it.  A wavefront with any other operand divides, and looks the
        // quotient up with scale 1; what lies outside [-1, 1] takes the first or last code, a NaN the last, as the search
        // does.  15.2 instead of 21.1 vector instructions an element over the whole kernel (14.3 instead of 20.5 for 16-bit types):
        // 26.2 M elements of the normal book 24.5 -> 21.3 us (fp32, 119
        // MB, 5.6 TB/s) and 19.9 -> 14.2 us (bf16), with two outliers 32.5 -> 27.5 and 30.0 -> 21.0; what is left of the
        // difference to the linear 4-bit pack kernel (19.6 and 13.0) is the table, 2 KiB copied per 2048 or 4096
        // elements (by workgroups half and a quarter as large: 25.8 and 29.4 us, fp32).
        const uint32_t scale_exponent = (as_u32(scale) >> 23) & 0xFFu;
        bool unusual = scale_exponent > 127u + 60u;
        if (any_nan) {   // wavefront-uniform
#pragma unroll
            for (int i = 0; i < VEC; ++i) unusual |= !(__builtin_fabsf(v[i]) <= scale);
        }
        float divisor = scale;
        if (__ballot(unusual) != 0) {   // wavefront-uniform
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const float t = v[i] / scale;
                v[i] = t < 1.0f ? (t > -1.0f ? t : -1.0f) : 1.0f;
            }
            divisor = 1.0f;
        }
        if constexpr (STOCHASTIC_BOOK) {
            // The quotient itself is wanted: how far it lies between two entries decides against the draw.  t = v / scale, the
            // IEEE quotient: a lane's elements share the divisor, so the reciprocal part of the division is done once
            // (v_rcp_f32 and one Newton step), then per element the product and two corrections.  These are the very
            // operations the compiler emits for `v / scale`, minus its operand scaling and special-case fix-up
            // (v_div_scale / v_div_fmas / v_div_fixup), which change nothing while the divisor lies in [2^-60, 2^60],
            // |v| <= scale, and the dividend is not so small (below 2^-103) that the division would rescale it; the
            // quotient is then below 2^-80, and no draw is below 2^-33.  tests/native/quotient_check.hip compares the
            // two forms on the device.  The entry below t is one table lookup and the fraction of the gap three operations: 26.2 M elements
            // of the normal book 27.1 us (fp32) and 23.2 (bf16), with a search in four halving steps and a division 37.6 and 34.7.
            float reciprocal = __builtin_amdgcn_rcpf(divisor);
            reciprocal = __builtin_fmaf(__builtin_fmaf(-divisor, reciprocal, 1.0f), reciprocal, reciprocal);
            uint32_t words[WORDS];
#pragma unroll
            for (int k = 0; k < WORDS; ++k) {
                uint32_t codes = 0;
#pragma unroll
                for (int i = 8 * k; i < 8 * k + 8; ++i) {
                    float t = v[i] * reciprocal;
                    t = __builtin_fmaf(__builtin_fmaf(-divisor, t, v[i]), reciprocal, t);
                    t = __builtin_fmaf(__builtin_fmaf(-divisor, t, v[i]), reciprocal, t);
                    const book_cells::Cell cell = table.cells[book_cells::nearest_place(t, 128.0f) - book_cells::kPlaceBits];
                    const uint32_t entry = cell.base + (t >= cell.threshold ? 1u : 0u);
                    const book_cells::Gap gap = table.gaps[entry];
                    const float fraction = book_cells::fraction_of_gap(t - gap.low, gap.gap, gap.reciprocal);
                    codes = (codes << 4) | (entry + (uniform[i] < fraction ? 1u : 0u));
                }
                words[k] = WIDE ? codes : __builtin_amdgcn_alignbit(codes, codes, 16);
            }
            if (live) store_words<WORDS, ITEM, kPlain>(group_codes + k0 * BIT / 8, words);
            store_meta();
            return;
        }
        const float reciprocal128 = __builtin_amdgcn_rcpf(divisor) * 128.0f, divisor24 = divisor * 0x1p-24f;
        if (live) {
            uint32_t words[WORDS];
#pragma unroll
            for (int k = 0; k < WORDS; ++k) {
                uint32_t codes = 0, below = 0;
#pragma unroll
                for (int i = 8 * k; i < 8 * k + 8; ++i) {
                    const book_cells::Cell cell = table.cells[book_cells::nearest_place(v[i], reciprocal128) - book_cells::kPlaceBits];
                    const float sign = book_cells::reaches(cell.threshold, v[i], divisor, divisor24);
                    codes = __builtin_amdgcn_alignbit(codes, cell.base, 28);          // (codes << 4) | code + 1
                    below = __builtin_amdgcn_alignbit(below, as_u32(sign), 28);
                }
                codes -= (below >> 3) & 0x11111111u;
                words[k] = WIDE ? codes : __builtin_amdgcn_alignbit(codes, codes, 16);
            }
            store_words<WORDS, ITEM, kPlain>(group_codes + k0 * BIT / 8, words);
        }
        store_meta();
        return;
    }

    int c[VEC];
    {
        const float multiplier = W::LEVELS / scale;
        constexpr int L = static_cast<int>(W::LEVELS);
        // Beside outliers and NaNs no magnitude exceeds the scale, so the product stays within the levels and adding
        // 1.5 * 2^23 leaves its rounding, half to even, in the low bits: two instructions an element instead of four
        // with conversion and clamp.  An outlier's code is cleared below; a NaN of a 16-bit type has zeros there.
        // With the search's keys and the clearing of words this took the kernel, bound by instructions, from 20.2 to
        // 17 us on 26.2 M bf16 elements with two outliers (the round trip 31.9 to 28.6).
        // With noise the product is clamped first, which a NaN would not survive as the 0 it encodes as: a wavefront that
        // holds one, or an infinite scale (infinity times the multiplier 0), rounds, converts and clamps.
        // nvcc contracts v * m + noise into one FMA; without noise the product is rounded alone
        auto scaled = [&](int i) { return STOCHASTIC ? __builtin_fmaf(v[i], multiplier, uniform[i] - 0.5f) : v[i] * multiplier; };
        if (!STOCHASTIC && (!WIDE || !any_nan)) {
#pragma unroll
            for (int i = 0; i < VEC; ++i) c[i] = static_cast<int>(as_u32(scaled(i) + 0x1.8p23f));
        } else if (STOCHASTIC && !any_nan && __ballot(scale_not_finite(scale)) == 0) {   // wavefront-uniform
#pragma unroll
            for (int i = 0; i < VEC; ++i)
                c[i] = static_cast<int>(as_u32(__builtin_amdgcn_fmed3f(scaled(i), -W::LEVELS, W::LEVELS) + 0x1.8p23f));
        } else {
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const int r = cvt_i32(__builtin_rintf(scaled(i)));
                c[i] = r < -L ? -L : (r > L ? L : r);
            }
        }
    }
    if (live) {
        uint32_t words[WORDS];
        if constexpr (BIT == 8) pack_codes<T, 8, VEC, WORDS>(c, words);
        else pack_nibbles<T, EL>(c, words);
        if constexpr (!(FIXED & 1)) {
            constexpr uint32_t PER_WORD = 32 / BIT, ORDER = BIT == 8 ? (WIDE ? 3 : 1) : (WIDE ? 7 : 3);   // place in a word
            uint32_t code[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) code[k] = ((1u << BIT) - 1) << (((outlier[k] ^ ORDER) * BIT) & 31u);
#pragma unroll
            for (uint32_t w = 0; w < WORDS; ++w)
                words[w] &= ~((outlier[0] / PER_WORD == w ? code[0] : 0u) | (outlier[1] / PER_WORD == w ? code[1] : 0u));
        }
        store_words<WORDS, ITEM, kPlain>(group_codes + k0 * BIT / 8, words);
    }
    store_meta();
}

// ---------------------------------------------------------------------------------------------
// dequantize (optionally combined into `out`)
// ---------------------------------------------------------------------------------------------
template <typename T, int G, int BIT>
__global__ __launch_bounds__(kBlock) void wire_general_decode_kernel(const WireGeneralDecodeArgs a) {
    using W = wire<T, BIT>;
    using Raw = typename raw_bits<T>::type;
    constexpr int VEC = W::VEC, ITEM = sizeof(T), CB = G * BIT / 8;

    const int lane = threadIdx.x & (kWave - 1);
    const int meta_bytes = meta_words_of(a.topk) * ITEM;
    const int64_t groups = a.numel / G;
    const int64_t tile_first = (static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6)) * W::TILE;
    if (tile_first >= a.numel) return;   // wavefront-uniform
    const int64_t e0 = tile_first + lane * VEC;
    const bool live = e0 < a.numel;      // dead lanes read group 0 and store nothing
    const int64_t group = live ? e0 / G : 0;
    const int k0 = live ? static_cast<int>(e0 - group * G) : 0;
    const uint8_t *group_codes = a.payload + (a.compact ? group * (CB + meta_bytes) : group * CB);
    const uint8_t *group_meta = a.compact ? group_codes + CB : a.payload + groups * CB + group * meta_bytes;

    uint32_t words[W::WORDS];
    load_piece<T, BIT, kPlain, W::WORDS>(group_codes + piece_offset<T, BIT>(k0), words);
    // the group's metadata words [scale][indices][top1][top2], fetched together with the codes
    Raw meta[4] = {0, 0, 0, 0};
    if (a.topk == 2) {
        load_elems<Raw, 4, kPlain>(reinterpret_cast<const Raw *>(group_meta), meta);
    } else if (a.topk == 1) {
        Raw pair[2];
        load_elems<Raw, 2, kPlain>(reinterpret_cast<const Raw *>(group_meta), pair);
        meta[0] = pair[0];
        meta[1] = pair[1];
        meta[2] = *reinterpret_cast<const Raw *>(group_meta + 2 * ITEM);
    } else {
        meta[0] = *reinterpret_cast<const Raw *>(group_meta);
    }
    const float scale = value_of<T>(meta[0]);
    const float *book = wave_code_book(a.kind, lane);   // after the loads were issued: its wait covers theirs
    const float step = a.kind == 0 ? step_of<BIT>(scale) : scale;

    Raw decoded[VEC];
    if (BIT == 4 && a.kind != 0) {   // uniform: the code's four bits, as they are, index the book
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            const int top = 16 - 16 * (i / 4) + 4 * (i % 4);   // left shift that puts the nibble on top, as in unpack_code
            decoded[i] = static_cast<Raw>(raw_from<T>(book[(words[0] << top) >> 28] * step));
        }
    } else {
#pragma unroll
        for (int i = 0; i < VEC; ++i)
            decoded[i] = static_cast<Raw>(raw_from<T>(unpack_code<T, BIT, W::WORDS>(words, i) * step));
    }
    if (a.topk >= 1) {
        const uint32_t indices = meta[1];
        const int index1 = static_cast<int>(indices & 0xFFu);
        const int index2 = a.topk == 2 ? static_cast<int>((indices >> 8) & 0xFFu) : -1;
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            if (k0 + i == index1) decoded[i] = meta[2];
            if (k0 + i == index2) decoded[i] = meta[3];   // written second, as in the reference
        }
    }
    if (!live) return;
    Raw *out = static_cast<Raw *>(a.out) + e0;
    if (a.op != 0) {
        Raw old[VEC];
        load_elems<Raw, VEC, kNonTemporal>(out, old);
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            const float o = value_of<T>(old[i]), d = value_of<T>(decoded[i]);
            if (a.op == 1) decoded[i] = static_cast<Raw>(raw_from<T>(add_in<T>(o, d)));
            else if (a.op == 2) decoded[i] = o > d ? old[i] : decoded[i];
            else decoded[i] = o > d ? decoded[i] : old[i];
        }
    }
    // The decoded tensor is the large stream of this kernel and nothing here reads it again: with the non-temporal
    // hint the decode of 26.2 M fp32 elements takes 19.9 instead of 30.2 us (top-2), 18.0 instead of 31.1 us (code book).
    store_elems<Raw, VEC, kNonTemporal>(out, decoded);
}

// The same with two tiles a wavefront, the loads of both issued before the first is decoded.  A text of its own because what the two
// could share costs the single tile: as one kernel for either number 1 to 2 % on 13 and 26 M fp32 elements, as two kernels that inline the
// same load and decode functions 5 to 6 % there (normal book, us of quantize + decode: 9 M 15.7 / 16.4, 26.2 M 38.7 / 41.1) and up to 3 % on
// small ones.  A change to either belongs in both; the tests compare them over codes, outliers and combining decodes.
template <typename T, int G, int BIT>
__global__ __launch_bounds__(kBlock) void wire_general_decode_pair_kernel(const WireGeneralDecodeArgs a) {
    constexpr int TILES = 2;
    using W = wire<T, BIT>;
    using Raw = typename raw_bits<T>::type;
    constexpr int VEC = W::VEC, ITEM = sizeof(T), CB = G * BIT / 8;

    const int lane = threadIdx.x & (kWave - 1);
    const int meta_bytes = meta_words_of(a.topk) * ITEM;
    const int64_t groups = a.numel / G;
    const int64_t first = (static_cast<int64_t>(blockIdx.x) * kWavesPerBlock * TILES + (threadIdx.x >> 6)) * W::TILE;
    if (first >= a.numel) return;   // wavefront-uniform
    uint32_t words[TILES][W::WORDS];
    Raw meta[TILES][4];
    int k0[TILES];
    bool live[TILES];      // dead lanes read group 0 and store nothing
    int64_t e0[TILES];
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
        e0[u] = first + u * kWavesPerBlock * W::TILE + lane * VEC;
        live[u] = e0[u] < a.numel;
        const int64_t group = live[u] ? e0[u] / G : 0;
        k0[u] = live[u] ? static_cast<int>(e0[u] - group * G) : 0;
        const uint8_t *group_codes = a.payload + (a.compact ? group * (CB + meta_bytes) : group * CB);
        const uint8_t *group_meta = a.compact ? group_codes + CB : a.payload + groups * CB + group * meta_bytes;
        load_piece<T, BIT, kPlain, W::WORDS>(group_codes + piece_offset<T, BIT>(k0[u]), words[u]);
        // the group's metadata words [scale][indices][top1][top2], fetched together with the codes
        meta[u][0] = meta[u][1] = meta[u][2] = meta[u][3] = 0;
        if (a.topk == 2) {
            load_elems<Raw, 4, kPlain>(reinterpret_cast<const Raw *>(group_meta), meta[u]);
        } else if (a.topk == 1) {
            Raw pair[2];
            load_elems<Raw, 2, kPlain>(reinterpret_cast<const Raw *>(group_meta), pair);
            meta[u][0] = pair[0];
            meta[u][1] = pair[1];
            meta[u][2] = *reinterpret_cast<const Raw *>(group_meta + 2 * ITEM);
        } else {
            meta[u][0] = *reinterpret_cast<const Raw *>(group_meta);
        }
    }
    float scale[TILES];
#pragma unroll
    for (int u = 0; u < TILES; ++u) scale[u] = value_of<T>(meta[u][0]);
    const float *book = wave_code_book(a.kind, lane);   // after the loads were issued: its wait covers theirs
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
        const float step = a.kind == 0 ? step_of<BIT>(scale[u]) : scale[u];
        Raw decoded[VEC];
        if (BIT == 4 && a.kind != 0) {   // uniform: the code's four bits, as they are, index the book
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const int top = 16 - 16 * (i / 4) + 4 * (i % 4);   // left shift that puts the nibble on top, as in unpack_code
                decoded[i] = static_cast<Raw>(raw_from<T>(book[(words[u][0] << top) >> 28] * step));
            }
        } else {
#pragma unroll
            for (int i = 0; i < VEC; ++i) decoded[i] = static_cast<Raw>(raw_from<T>(unpack_code<T, BIT, W::WORDS>(words[u], i) * step));
        }
        if (a.topk >= 1) {
            const uint32_t indices = meta[u][1];
            const int index1 = static_cast<int>(indices & 0xFFu);
            const int index2 = a.topk == 2 ? static_cast<int>((indices >> 8) & 0xFFu) : -1;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                if (k0[u] + i == index1) decoded[i] = meta[u][2];
                if (k0[u] + i == index2) decoded[i] = meta[u][3];   // written second, as in the reference
            }
        }
        if (!live[u]) continue;
        Raw *out = static_cast<Raw *>(a.out) + e0[u];
        if (a.op != 0) {
            Raw old[VEC];
            load_elems<Raw, VEC, kNonTemporal>(out, old);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const float o = value_of<T>(old[i]), d = value_of<T>(decoded[i]);
                if (a.op == 1) decoded[i] = static_cast<Raw>(raw_from<T>(add_in<T>(o, d)));
                else if (a.op == 2) decoded[i] = o > d ? old[i] : decoded[i];
                else decoded[i] = o > d ? decoded[i] : old[i];
            }
        }
        // The decoded tensor is the large stream of this kernel and nothing here reads it again: with the non-temporal
        // hint the decode of 26.2 M fp32 elements takes 19.9 instead of 30.2 us (top-2), 18.0 instead of 31.1 us (code book);
        // written through as well it loses 1 to 6 %.
        store_elems<Raw, VEC, kNonTemporal>(out, decoded);
    }
}

template <typename T, int G, int BIT, int FIXED, int EL>
hipError_t launch_general_quant_as(const WireGeneralQuantArgs &a, hipStream_t stream) {
    const int64_t tile = static_cast<int64_t>(kWave) * EL * kWavesPerBlock;
    const int64_t blocks = (a.numel + tile - 1) / tile;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    hipLaunchKernelGGL((wire_general_quant_kernel<T, G, BIT, FIXED, EL>), grid, dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

template <typename T, int G>
hipError_t launch_general_quant_g(int bit, const WireGeneralQuantArgs &a, hipStream_t stream) {
    // Every policy runs a kernel without the code of the others.  us for 26.2 M elements in groups of 64 with the codes apart, fp32
    // and bf16 (launches alone, in rotation over 1 GB): top-2 25.2 and 17.0, stochastic 24.0 and 16.6, the two together 29.3 and
    // 21.6, 4-bit top-2 23.0 and 15.6, a code book 21.3 and 14.2, with outliers 26.0 and 19.1, rounded stochastically 27.1 and
    // 23.2, with outliers 36.3 and 29.3.  (As one kernel for every policy top-2 took 28.5 and 24.2, stochastic 24.0 and
    // 21.8, the two together 33.9 and 27.0: for sixteen 16-bit elements a lane it held four wavefronts a SIMD, the one for
    // plain stochastic codes holds eight.)
    //
    // One tile of 32 bytes a lane a wavefront.  Two such tiles, both asked for before either is encoded: top-2 29.9 against
    // 26.7 us (fp32) and 21.0 against 17.4 (bf16), a code book 22.0 against 21.3 and 14.7 against 14.2.  16 bytes a lane
    // for 16-bit types: a code book 15.7, two tiles of top-2 22.0; 64 bytes: top-2 17.7, and 26.9 (fp32).
    constexpr int WIDE = general_quant_elems<T>() <= G ? general_quant_elems<T>() : G;
    if (bit != 8 && bit != 4) return hipErrorNotSupported;
    if (bit == 8 && a.kind != 0) return hipErrorNotSupported;   // eight bits: linear codes only
    // plain linear codes: lbc_wire_quant_pack serves those calls, and no kernel here has their code
    if (a.kind == 0 && a.topk == 0 && !a.stochastic) return hipErrorNotSupported;
    if (bit == 8) {
        if (a.stochastic && a.topk == 0) return launch_general_quant_as<T, G, 8, 13, WIDE>(a, stream);
        if (a.stochastic) return launch_general_quant_as<T, G, 8, 12, WIDE>(a, stream);
        return launch_general_quant_as<T, G, 8, 6, WIDE>(a, stream);
    }
    if (a.kind == 0) {
        if (a.stochastic && a.topk == 0) return launch_general_quant_as<T, G, 4, 13, WIDE>(a, stream);
        if (a.stochastic) return launch_general_quant_as<T, G, 4, 12, WIDE>(a, stream);
        return launch_general_quant_as<T, G, 4, 6, WIDE>(a, stream);
    }
    if (a.stochastic && a.topk == 0) return launch_general_quant_as<T, G, 4, 9, WIDE>(a, stream);
    if (a.stochastic) return launch_general_quant_as<T, G, 4, 8, WIDE>(a, stream);
    if (a.topk == 0) return launch_general_quant_as<T, G, 4, 3, WIDE>(a, stream);
    return launch_general_quant_as<T, G, 4, 2, WIDE>(a, stream);
}

template <typename T> hipError_t launch_general_quant_t(int g, int bit, const WireGeneralQuantArgs &a, hipStream_t s) {
    switch (g) {
        case 64: return launch_general_quant_g<T, 64>(bit, a, s);
        case 32: return launch_general_quant_g<T, 32>(bit, a, s);
        case 16: return launch_general_quant_g<T, 16>(bit, a, s);
        default: return hipErrorNotSupported;
    }
}

// The decode waits for short loads, the codes and a group's words, so beyond the chip's wavefront slots two tiles a wavefront pay: in 16
// bits where there is a code book or an outlier to wait for as well, in fp32 with two outliers, or up to 3 Mi elements without one and
// 4 Mi with one.  us of quantize + decode with one / two tiles, three tensors in rotation (and beyond the last-level cache): two outliers
// fp32 8-bit 3 Mi 9.4 / 9.0 (10.0 / 9.5), 6.25 Mi 14.6 / 14.1 (15.9 / 15.6), e2m1 25 Mi 48.5 / 47.4 (47.0 / 46.3), bf16 8-bit 5 Mi 9.9 / 9.3 (10.4 / 9.8),
// 25 Mi 29.1 / 28.2 (30.5 / 29.9); one outlier bf16 6.25 Mi 11.3 / 10.9 (11.8 / 11.4), fp32 3 Mi 9.1 / 8.9 (9.7 / 9.4), 4.6 M 12.4 / 13.0 (13.6 / 14.2),
// 20 Mi 36.3 / 36.3 (37.4 / 37.6); none, normal book bf16 6.25 Mi 10.3 / 9.7 (10.9 / 10.5), 25 Mi 24.9 / 24.7 (26.9 / 26.6), fp32 2.7 M 7.8 / 7.5 (8.4 /
// 8.3), 4.7 M 10.6 / 11.3 (11.8 / 12.6), 6.6 M 12.7 / 12.9 (13.8 / 14.1), linear bf16 8 Mi 15.2 / 15.5 (15.2 / 15.4).
template <typename T, int G, int BIT>
hipError_t launch_general_decode_b(const WireGeneralDecodeArgs &a, hipStream_t stream) {
    const bool fills = a.numel > kResidentWaves * wire<T, BIT>::TILE;
    const bool waits = sizeof(T) == 2 ? a.topk > 0 || a.kind != 0 : a.topk == 2 || a.numel <= static_cast<int64_t>(3 + a.topk) << 20;
    const bool pair = fills && waits;
    const int64_t tile = wire<T, BIT>::TILE * kWavesPerBlock * (pair ? 2 : 1);
    const int64_t blocks = (a.numel + tile - 1) / tile;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    if (pair) hipLaunchKernelGGL((wire_general_decode_pair_kernel<T, G, BIT>), grid, dim3(kBlock), 0, stream, a);
    else hipLaunchKernelGGL((wire_general_decode_kernel<T, G, BIT>), grid, dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

template <typename T, int G>
hipError_t launch_general_decode_g(int bit, const WireGeneralDecodeArgs &a, hipStream_t stream) {
    if (bit == 8) return launch_general_decode_b<T, G, 8>(a, stream);
    if (bit == 4) return launch_general_decode_b<T, G, 4>(a, stream);
    return hipErrorNotSupported;
}

template <typename T> hipError_t launch_general_decode_t(int g, int bit, const WireGeneralDecodeArgs &a, hipStream_t s) {
    switch (g) {
        case 64: return launch_general_decode_g<T, 64>(bit, a, s);
        case 32: return launch_general_decode_g<T, 32>(bit, a, s);
        case 16: return launch_general_decode_g<T, 16>(bit, a, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace

hipError_t launch_wire_general_quant(int dtype, int group_size, int bit, const WireGeneralQuantArgs &args,
                                     hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_general_quant_t<float>(group_size, bit, args, stream);
        case kF16: return launch_general_quant_t<f16>(group_size, bit, args, stream);
        case kBF16: return launch_general_quant_t<bf16>(group_size, bit, args, stream);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_wire_general_decode(int dtype, int group_size, int bit, const WireGeneralDecodeArgs &args,
                                      hipStream_t stream) {
    switch (dtype) {
        case kF32: return launch_general_decode_t<float>(group_size, bit, args, stream);
        case kF16: return launch_general_decode_t<f16>(group_size, bit, args, stream);
        case kBF16: return launch_general_decode_t<bf16>(group_size, bit, args, stream);
        default: return hipErrorNotSupported;
    }
}

}  // namespace lbc
