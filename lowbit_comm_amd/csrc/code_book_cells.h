// The 4-bit code books of the reference's CUDA extension (ccdl_comm/csrc/quantization/inner.cuh:9-35) and, built
// from them at compile time, a one-lookup form of its encoder.
//
// The reference encodes t = v / scale by a search for the largest entry not above t followed by a rounding step,
// `entry + (t - book[entry] > (book[entry + 1] - book[entry]) * 0.5f)` (inner.cuh:74-118).  For one book that is a
// non-decreasing step function of t with fourteen steps.  The places of the steps (the smallest float at which the
// code becomes k + 1) are found here by bisection over the float line with the reference's own arithmetic, and
// [-1, 1] is cut into 256 cells of width 1/128.  A cell stores the code at its left end and the next step from there
// on, inside the cell or beyond it, so that
//     code(t) = cell.base + (t >= cell.threshold),   cell = cells[(unsigned)fma(t, 128, 128)]
// for every finite t in [-1, 1].  tests/native/check_book_cells.cpp compares the two forms on every such float on the host,
// tests/native/book_cells_check.hip what the quantize kernel makes of them (below) on the device.
//
// The quantize kernel does not form t.  Steps lie at least two cells apart, so a cell answers for every t from its left
// end to one and a half cells behind it: the cell one below the rounded place of an approximate quotient (`nearest_place`)
// is right for any error up to a quarter of a cell.  Whether the quotient, rounded to a float, reaches
// the step is then decided without a division (`reaches`).
// Plain C++17 (host and device): no HIP types.
#pragma once
#include <cstdint>

namespace lbc {
namespace book_cells {

constexpr int kBooks = 4;
constexpr int kCells = 257;   // (unsigned)(t * 128 + 128) for t in [-1, 1] is 0..256

// entry 15 is never produced by the encoder
struct Books {
    float value[kBooks][16];
};
constexpr Books kBookSet = {{
    {-1.0f, -0.815410147f, -0.655160150f, -0.510228027f, -0.375324982f, -0.246951370f, -0.122538030f, 0.0f,
     0.122538030f, 0.246951370f, 0.375324982f, 0.510228027f, 0.655160150f, 0.815410147f, 1.0f, __builtin_inff()},
    {-1.0f, -0.85714286f, -0.71428571f, -0.57142857f, -0.42857143f, -0.28571429f, -0.14285714f, 0.0f,
     0.14285714f, 0.28571429f, 0.42857143f, 0.57142857f, 0.71428571f, 0.85714286f, 1.0f, __builtin_inff()},
    {-1.0f, -0.5f, -0.25f, -0.125f, -0.0625f, -0.03125f, -0.015625f, 0.0f,
     0.015625f, 0.03125f, 0.0625f, 0.125f, 0.25f, 0.5f, 1.0f, __builtin_inff()},
    {-1.0f, -0.6666666666666666f, -0.5f, -0.3333333333333333f, -0.25f, -0.16666666666666666f, -0.125f, 0.0f,
     0.125f, 0.16666666666666666f, 0.25f, 0.3333333333333333f, 0.5f, 0.6666666666666666f, 1.0f, __builtin_inff()},
}};

struct alignas(8) Cell {   // the kernel copies it as two dwords
    float threshold;   // the code rises by one at this value, the next step at or behind the left end; +inf behind the last
    uint32_t base;     // the code at the cell's left end
};
struct Table {
    Cell cell[kCells];
};
struct Tables {
    Table book[kBooks];
};

// The reference's encoder for a number t (not NaN): search, then rounding.
constexpr int searched_code(const float (&book)[16], float t) {
    int at = 0;
    for (int entry = 1; entry <= 14; ++entry)
        if (!(t < book[entry])) at = entry;
    if (at == 14) return 14;   // the gap to entry 15 is infinite: never rounds up
    const float low = book[at], gap = book[at + 1] - low, excess = t - low;
    return at + (excess > gap * 0.5f ? 1 : 0);
}

// Floats as unsigned keys in the order of their values, and back.
constexpr uint32_t key_of(float f) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, f);
    return (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
}
constexpr float float_of(uint32_t key) {
    return __builtin_bit_cast(float, (key & 0x80000000u) ? (key & 0x7FFFFFFFu) : ~key);
}

// t * 128 is exact, so this is the device's single-rounding fma(t, 128, 128).
constexpr int cell_of(float t) { return static_cast<int>(t * 128.0f + 128.0f); }

// The smallest float in [-1, 1] whose code is above k.
constexpr float step_after(const float (&book)[16], int k) {
    uint32_t below = key_of(-1.0f), reached = key_of(1.0f);   // code(-1) = 0 <= k < 14 = code(1)
    while (reached - below > 1) {
        const uint32_t middle = below + (reached - below) / 2;
        if (searched_code(book, float_of(middle)) > k) reached = middle;
        else below = middle;
    }
    return float_of(reached);
}

constexpr Table make_table(const float (&book)[16]) {
    Table table{};
    float step[14]{};
    for (int k = 0; k < 14; ++k) step[k] = step_after(book, k);
    for (int i = 0; i < kCells; ++i) {
        uint32_t base = 0;
        float threshold = __builtin_inff();
        for (int k = 0; k < 14; ++k) {
            if (cell_of(step[k]) < i) ++base;
            else if (step[k] < threshold) threshold = step[k];
        }
        table.cell[i] = Cell{threshold, base};
    }
    return table;
}

// Steps at least two cells apart (up to a unit in the last place): see nearest_place.  None is a positive power of two,
// which would be closer to the float before it than its exponent says: see reaches.
constexpr bool steps_far_apart(const float (&book)[16]) {
    for (int k = 0; k < 14; ++k) {
        const float step = step_after(book, k);
        if (k > 0 && (step - step_after(book, k - 1)) * 128.0f < 1.999f) return false;
        if (step > 0.0f && (__builtin_bit_cast(uint32_t, step) & 0x007FFFFFu) == 0) return false;
    }
    return true;
}

constexpr Tables kTables = {{make_table(kBookSet.value[0]), make_table(kBookSet.value[1]), make_table(kBookSet.value[2]),
                               make_table(kBookSet.value[3])}};
static_assert(steps_far_apart(kBookSet.value[0]) && steps_far_apart(kBookSet.value[1]) &&
                  steps_far_apart(kBookSet.value[2]) && steps_far_apart(kBookSet.value[3]),
              "two steps of a code book lie too close for one lookup");

// The lookup of a quotient t.  No kernel runs it: the kernel's tables below are made from these cells, and
// tests/native/check_book_cells.cpp holds them against the search.
constexpr int cell_code(const Table &table, float t) {
    const Cell &cell = table.cell[cell_of(t)];
    return static_cast<int>(cell.base) + (t >= cell.threshold ? 1 : 0);
}

// ---- the lookup of v / scale without the quotient ----
#if defined(__HIPCC__)
#define LBC_CELLS_HOST_DEVICE __attribute__((host)) __attribute__((device)) __attribute__((always_inline)) inline
#else
#define LBC_CELLS_HOST_DEVICE inline
#endif

constexpr float kBeyond = 3.0f;   // no quotient of at most 1 reaches it

// The cells as the quantize kernel reads them, by place: entry p is the cell one below p, kBeyond stands behind the last
// step, and the code plus one lies in the top four bits, from where a funnel shift pushes it into a word of codes.
struct Places {
    Cell entry[kBooks][kCells];
};
constexpr Places make_places() {
    Places places{};
    for (int b = 0; b < kBooks; ++b)
        for (int p = 0; p < kCells; ++p) {
            const Cell &cell = kTables.book[b].cell[p == 0 ? 0 : p - 1];
            places.entry[b][p] = Cell{cell.threshold < kBeyond ? cell.threshold : kBeyond, (cell.base + 1) << 28};
        }
    return places;
}
constexpr Places kPlaces = make_places();

// ---- stochastic rounding: the largest entry not above t, its gap to the next one and that gap's reciprocal ----
// The same cells over the entries 1 .. 14 instead of the steps (they lie two cells apart or more as well): by place, `base` the
// count of entries passed.
constexpr Places make_floors() {
    Places places{};
    for (int b = 0; b < kBooks; ++b)
        for (int p = 0; p < kCells; ++p) {
            const int cell = p == 0 ? 0 : p - 1;
            uint32_t base = 0;
            float threshold = kBeyond;
            for (int k = 1; k <= 14; ++k) {
                const float entry = kBookSet.value[b][k];
                if (entry * 128.0f + 128.0f < static_cast<float>(cell)) ++base;
                else if (entry < threshold) threshold = entry;
            }
            places.entry[b][p] = Cell{threshold, base};
        }
    return places;
}
constexpr Places kFloors = make_floors();
constexpr bool entries_far_apart(const float (&book)[16]) {
    for (int k = 1; k < 14; ++k)
        if ((book[k + 1] - book[k]) * 128.0f < 1.999f) return false;
    return true;
}
static_assert(entries_far_apart(kBookSet.value[0]) && entries_far_apart(kBookSet.value[1]) &&
                  entries_far_apart(kBookSet.value[2]) && entries_far_apart(kBookSet.value[3]),
              "two entries of a code book lie too close for one lookup");

// Entry 14 is the last that the search gives and 1 the largest t: its gap, infinite in the book, only has to keep the
// fraction (t - 1) / gap from being positive.
struct alignas(16) Gap {   // the kernel copies it as four dwords
    float low, gap, reciprocal, unused;
};
struct Gaps {
    Gap entry[kBooks][16];
};
constexpr Gaps make_gaps() {
    Gaps gaps{};
    for (int b = 0; b < kBooks; ++b)
        for (int k = 0; k < 16; ++k) {
            const float low = kBookSet.value[b][k < 15 ? k : 14], gap = k < 14 ? kBookSet.value[b][k + 1] - low : 1.0f;
            gaps.entry[b][k] = Gap{low, gap, 1.0f / gap, 0.0f};
        }
    return gaps;
}
constexpr Gaps kGaps = make_gaps();

// The place of v / scale, round(128 * v / scale) + 128, in the low bits of a float: adding 1.5 * 2^23 + 128 rounds to an
// integer.  `reciprocal128` is 128 / scale with a few ulps of error.
constexpr float kPlaceMagic = 12582912.0f + 128.0f;
constexpr uint32_t kPlaceBits = 0x4B400000u;   // bits of 1.5 * 2^23: place 0
LBC_CELLS_HOST_DEVICE uint32_t nearest_place(float v, float reciprocal128) {
    return __builtin_bit_cast(uint32_t, __builtin_fmaf(v, reciprocal128, kPlaceMagic));
}

// A number whose sign bit is clear when RN(v / scale) >= threshold and set when it is below, for a scale of at least
// 2^-20.  The quotient rounds up to the threshold when it lies above m, the middle between the threshold and the float
// before it: m = threshold - h, with h half a unit in the threshold's last place (no threshold is a positive power of two, so the
// float before it has the same exponent).  It never equals m: m has 25 significant bits, so m * scale has at least 25 and
// is no float.  With b = v - threshold * scale, exactly, what counts is the sign of b + h * scale.  The inner operation
// gives b exactly while |b| <= 2 h scale (b is then a multiple of 2^-24 of its bound: v, being near threshold * scale,
// is a coarser multiple than the product), otherwise a rounded b on the same side of -h * scale; the outer one adds
// h * scale, whose power of two is threshold's exponent times 2^-24 (`scale24` is scale * 2^-24, exact).  (An infinite threshold
// would meet itself here: kBeyond.)
LBC_CELLS_HOST_DEVICE float reaches(float threshold, float v, float scale, float scale24) {
    const float b = __builtin_fmaf(-threshold, scale, v);
    const float exponent = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, threshold) & 0xFF800000u);
    return __builtin_fmaf(__builtin_fabsf(exponent), scale24, b);
}

// excess / gap for a gap of the books, as the division rounds it: the product with the reciprocal and one correction
// (Markstein).  tests/native/check_book_quotients.cpp compares the two for every significand of the dividend and every gap; a
// quotient that underflows on the way is below 2^-100, and no draw is.
LBC_CELLS_HOST_DEVICE float fraction_of_gap(float excess, float gap, float reciprocal) {
    const float q = excess * reciprocal;
    return __builtin_fmaf(__builtin_fmaf(-q, gap, excess), reciprocal, q);
}
}  // namespace book_cells
}  // namespace lbc
