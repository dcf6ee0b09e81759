// Host check of the code-book encoder's lookup without a quotient (lowbit_comm_amd/csrc/code_book_cells.h: the place of
// an approximate quotient, then the sign of `reaches`) against the search-and-round form on the IEEE quotient v / scale
// (ccdl_comm/csrc/quantization/inner.cuh:74-118).  For each book and many scales: the dividends next to every step times
// the scale, dividends on the cells' ends, 8- and 11-bit dividends and scales, and random ones; each with reciprocals a
// few ulps to either side.  Build: g++ -O2 -std=c++17 -ffp-contract=off.  Prints "MISMATCHES n".
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../lowbit_comm_amd/csrc/code_book_cells.h"

namespace bc = lbc::book_cells;

static int searched(const float *book, float t) {
    int at = 0;
    for (int step = 8; step >= 1; step >>= 1) {
        const int mid = at + step;
        if (mid < 15 && !(t < book[mid])) at = mid;
    }
    const volatile float low = book[at];
    const volatile float gap = book[at + 1] - low;
    const volatile float excess = t - low;
    return at + (excess > gap * 0.5f ? 1 : 0);
}

static unsigned long long checked = 0, mismatches = 0;

static void check(int b, float v, float scale) {
    if (!(std::fabs(v) <= scale)) return;
    const volatile float t = v / scale;
    const int want = searched(bc::kBookSet.value[b], t);
    float reciprocal = 1.0f / scale;
    for (int ulps = -2; ulps <= 2; ++ulps) {
        const float r = bc::float_of(bc::key_of(reciprocal) + ulps) * 128.0f;
        const uint32_t place = bc::nearest_place(v, r) - bc::kPlaceBits;
        if (place >= static_cast<uint32_t>(bc::kCells)) {
            ++mismatches;
            continue;
        }
        const bc::Cell &cell = bc::kPlaces.entry[b][place];
        const float sign = bc::reaches(cell.threshold, v, scale, scale * 0x1p-24f);
        const int got = static_cast<int>(cell.base >> 28) - (std::signbit(sign) ? 1 : 0);
        mismatches += got != want;
        ++checked;
    }
}

// Stochastic rounding: the entry below t by the cells against the search, on every float of a stride and next to every
// entry; the fraction of the gap against the division, for every significand of the dividend and every gap.
static void check_floors() {
    for (int b = 0; b < bc::kBooks; ++b) {
        const float *book = bc::kBookSet.value[b];
        auto floor_of = [&](float t) {
            int at = 0;
            for (int step = 8; step >= 1; step >>= 1) {
                const int mid = at + step;
                if (mid < 15 && !(t < book[mid])) at = mid;
            }
            return at;
        };
        auto one = [&](float t) {
            if (!(std::fabs(t) <= 1.0f)) return;
            const bc::Cell &cell = bc::kFloors.entry[b][bc::nearest_place(t, 128.0f) - bc::kPlaceBits];
            mismatches += static_cast<int>(cell.base) + (t >= cell.threshold ? 1 : 0) != floor_of(t);
            ++checked;
        };
        for (uint32_t key = bc::key_of(-1.0f); key <= bc::key_of(1.0f); key += 509) one(bc::float_of(key));
        for (int k = 0; k < 15; ++k)
            for (int d = -4; d <= 4; ++d) one(bc::float_of(bc::key_of(book[k]) + d));
        for (int place = -256; place <= 256; ++place)
            for (int d = -2; d <= 2; ++d) one(bc::float_of(bc::key_of(place / 256.0f) + d));
        for (int k = 0; k < 14; ++k) {
            const bc::Gap &g = bc::kGaps.entry[b][k];
            if (g.low != book[k] || g.gap != book[k + 1] - book[k]) ++mismatches;
            unsigned long long bad = 0;
            for (uint32_t m = 0; m < (1u << 23); ++m) {
                const float excess = bc::float_of(0x80000000u | (120u << 23) | m);
                bad += bc::fraction_of_gap(excess, g.gap, g.reciprocal) != excess / g.gap;
            }
            mismatches += bad;
            checked += 1u << 23;
        }
    }
}

int main(int argc, char **argv) {
    check_floors();
    const int scales = argc > 1 ? std::atoi(argv[1]) : 20000;
    std::mt19937_64 rng(17);
    for (int i = 0; i < scales; ++i) {
        int exponent = static_cast<int>(rng() % 81) - 20;            // 2^-20 .. 2^60, with the mantissa the kernel's range
        uint32_t mantissa = static_cast<uint32_t>(rng()) & 0x7FFFFFu;
        const int kind = i % 4;                                       // all bits, 8 significant ones, 11, few (exact quotients)
        if (kind == 1) mantissa &= 0x7F0000u;
        if (kind == 2) mantissa &= 0x7FE000u;
        if (kind == 3) mantissa &= 0x700000u;
        float scale = bc::float_of(0x80000000u | (static_cast<uint32_t>(exponent + 127) << 23) | mantissa);
        if (scale < 1.0e-6f) scale = 1.0e-6f;
        for (int b = 0; b < bc::kBooks; ++b) {
            auto around = [&](float v, int reach) {
                for (int d = -reach; d <= reach; ++d) check(b, bc::float_of(bc::key_of(v) + d), scale);
            };
            for (int k = 0; k < 14; ++k) {
                const float near = bc::step_after(bc::kBookSet.value[b], k) * scale;
                around(near, 3);
                const uint32_t bits = __builtin_bit_cast(uint32_t, near);
                for (uint32_t keep : {0xFFFF0000u, 0xFFFFE000u})      // dividends of a 16-bit type
                    for (int d = -1; d <= 1; ++d) {
                        const uint32_t cut = (bits & keep) + static_cast<uint32_t>(d) * (~keep + 1);
                        check(b, __builtin_bit_cast(float, cut), scale);
                    }
            }
            for (int place = -128; place <= 128; place += 1 + static_cast<int>(rng() % 9)) around(place / 128.0f * scale, 1);
            around((static_cast<float>(rng() % 256) - 127.5f) / 128.0f * scale, 2);
            for (int n = 0; n < 8; ++n) check(b, static_cast<float>(static_cast<double>(rng()) * 0x1p-63 - 1.0) * scale, scale);
            check(b, 0.0f, scale);
            check(b, -0.0f, scale);
            check(b, scale, scale);
            check(b, -scale, scale);
        }
    }
    std::printf("CHECKED %llu\nMISMATCHES %llu\n", checked, mismatches);
    return mismatches ? 1 : 0;
}
