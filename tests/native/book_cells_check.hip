// Device check of the code-book lookups as the quantize kernel runs them (lowbit_comm_amd/csrc/code_book_cells.h), against the
// search and rounding that they stand for (ccdl_comm/csrc/quantization/inner.cuh:74-118), both evaluated on the device.  Rounded to
// nearest, without a quotient: the place of v * rcp(scale) with the hardware's own reciprocal, then the sign of `reaches`; for
// scale 1 and every float v in [-1, 1], and for scales of every exponent that the kernel takes this way (1e-6 .. 2^61) with
// dividends next to every step, next to the cells' ends and middles, in 8 and 11 significant bits, small and random.  Rounded
// stochastically: the entry below t and the fraction of the gap, for every float t in [-1, 1].  Prints "MISMATCHES n"; exit
// status 1 when n is not 0.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../lowbit_comm_amd/csrc/code_book_cells.h"

namespace bc = lbc::book_cells;

struct Steps {
    float at[bc::kBooks][14];
};
constexpr Steps make_steps() {
    Steps steps{};
    for (int b = 0; b < bc::kBooks; ++b)
        for (int k = 0; k < 14; ++k) steps.at[b][k] = bc::step_after(bc::kBookSet.value[b], k);
    return steps;
}

__constant__ bc::Books kBooks = bc::kBookSet;
__constant__ bc::Places kPlaces = bc::kPlaces, kFloors = bc::kFloors;
__constant__ bc::Gaps kGaps = bc::kGaps;
__constant__ Steps kSteps = make_steps();

__device__ int floor_of(const float *book, float t) {
    int at = 0;
    for (int step = 8; step >= 1; step >>= 1) {
        const int mid = at + step;
        if (mid < 15 && !(t < book[mid])) at = mid;
    }
    return at;
}

// 1 when the two forms differ, 0 when they agree or the kernel would not take v / scale this way
__device__ unsigned nearest_differs(int b, float v, float scale) {
    if (!(__builtin_fabsf(v) <= scale)) return 0;
    const float *book = kBooks.value[b];
    const float t = v / scale;
    const int at = floor_of(book, t);
    const float low = book[at], gap = book[at + 1] - low, excess = t - low;
    const int searched = at + (excess > gap * 0.5f ? 1 : 0);
    const uint32_t place = bc::nearest_place(v, __builtin_amdgcn_rcpf(scale) * 128.0f) - bc::kPlaceBits;
    if (place >= static_cast<uint32_t>(bc::kCells)) return 1;
    const bc::Cell cell = kPlaces.entry[b][place];
    const float sign = bc::reaches(cell.threshold, v, scale, scale * 0x1p-24f);
    return static_cast<int>(cell.base >> 28) - static_cast<int>(__float_as_uint(sign) >> 31) != searched;
}

__global__ void every_quotient(int b, uint32_t first_key, uint64_t count, unsigned long long *bad) {
    const float *book = kBooks.value[b];
    unsigned long long mine = 0;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x) {
        const float t = bc::float_of(first_key + (uint32_t)i);
        mine += nearest_differs(b, t, 1.0f);
        const int want = floor_of(book, t);
        const uint32_t place = bc::nearest_place(t, 128.0f) - bc::kPlaceBits;
        if (place >= static_cast<uint32_t>(bc::kCells)) {
            ++mine;
            continue;
        }
        const bc::Cell cell = kFloors.entry[b][place];
        const uint32_t entry = cell.base + (t >= cell.threshold ? 1u : 0u);
        if (entry != static_cast<uint32_t>(want)) {
            ++mine;
            continue;
        }
        const bc::Gap gap = kGaps.entry[b][entry];
        const float fraction = bc::fraction_of_gap(t - gap.low, gap.gap, gap.reciprocal);
        const float divided = (t - book[want]) / (book[want + 1] - book[want]);
        // no draw is below 2^-33: smaller fractions, and the last entry's zero, only have to stay below that
        mine += divided < 0x1p-90f ? !(fraction < 0x1p-90f) : fraction != divided;
    }
    if (mine) atomicAdd(bad, mine);
}

__device__ uint64_t next(uint64_t &state) {   // splitmix64
    uint64_t z = state += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void many_scales(int b, uint32_t scales, unsigned long long *counts) {
    unsigned long long mine = 0, seen = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < scales; i += gridDim.x * blockDim.x) {
        uint64_t state = i * 0xD1342543DE82EF95ull + b;
        const int exponent = static_cast<int>(i % 81u) - 20;                  // 2^-20 .. 2^60
        uint32_t mantissa = static_cast<uint32_t>(next(state)) & 0x7FFFFFu;
        const uint32_t kind = i / 81u % 4u;                                   // all bits, 8, 11 and 4 significant ones
        if (kind == 1) mantissa &= 0x7F0000u;
        if (kind == 2) mantissa &= 0x7FE000u;
        if (kind == 3) mantissa &= 0x700000u;
        float scale = __uint_as_float(static_cast<uint32_t>(exponent + 127) << 23 | mantissa);
        scale = scale < 1.0e-6f ? 1.0e-6f : scale;
        auto around = [&](float v, int reach) {
            for (int d = -reach; d <= reach; ++d) mine += nearest_differs(b, bc::float_of(bc::key_of(v) + d), scale);
            seen += 2 * reach + 1;
        };
        for (int k = 0; k < 14; ++k) {
            const float near = kSteps.at[b][k] * scale;
            around(near, 3);
            for (int bits = 16; bits >= 13; bits -= 3) {                      // dividends of a 16-bit type
                const uint32_t keep = ~0u << bits, unit = 1u << bits;
                for (int d = -1; d <= 1; ++d) mine += nearest_differs(b, __uint_as_float((__float_as_uint(near) & keep) + d * unit), scale);
                seen += 3;
            }
        }
        for (int half = -256; half <= 256; ++half) around(half / 256.0f * scale, 2);   // ends and middles of the cells
        for (int n = 0; n < 64; ++n) {
            const float unit = static_cast<float>(static_cast<int64_t>(next(state))) * 0x1p-63f;
            around(n & 1 ? unit * scale : __builtin_ldexpf(unit * scale, -static_cast<int>(next(state) % 160u)), 0);
        }
        around(0.0f, 1);
        around(scale, 0);
        around(-scale, 0);
    }
    if (mine) atomicAdd(counts, mine);
    atomicAdd(counts + 1, seen);
}

int main() {
    unsigned long long *counts, total = 0, checked = 0;
    if (hipMalloc(&counts, 2 * sizeof(*counts)) != hipSuccess) return 2;
    const uint32_t first = bc::key_of(-1.0f), last = bc::key_of(1.0f);
    const uint64_t count = (uint64_t)last - first + 1;
    for (int b = 0; b < bc::kBooks; ++b) {
        unsigned long long h[2] = {0, 0};
        if (hipMemcpy(counts, h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess) return 2;
        hipLaunchKernelGGL(every_quotient, dim3(8192), dim3(256), 0, 0, b, first, count, counts);
        hipLaunchKernelGGL(many_scales, dim3(1024), dim3(256), 0, 0, b, 1u << 18, counts);
        if (hipDeviceSynchronize() != hipSuccess) return 2;
        if (hipMemcpy(h, counts, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 2;
        printf("book %d: %llu quotients, %llu dividends, %llu mismatches\n", b, (unsigned long long)count, h[1], h[0]);
        total += h[0];
        checked += 2 * count + h[1];
    }
    printf("CHECKED %llu\nMISMATCHES %llu\n", checked, total);
    return total ? 1 : 0;
}
