// Group-wise INT8 quantize + pack for gfx950, optionally fused with the
// error-feedback compensate (x + r) and residual update (p - restored).
//
// Mapping.  One lane owns VEC consecutive elements, so a group of G elements
// sits in G/VEC adjacent lanes of one 16-lane DPP row and the group absmax is a
// DPP butterfly with no LDS.  VEC is chosen so that the widest stream of the
// call moves 16 bytes per lane per instruction: 4 when any fp32 tensor takes
// part (input, residual, restored), 8 for a pure 16-bit call.  A wavefront
// instruction then touches one contiguous run (1 KiB for the 16-byte streams);
// a 256-thread block walks UNROLL * 4 such tiles with all loads issued before
// the first use.  Codes leave as one 4-/8-byte store per lane, the scale as one
// float from the first lane of each group.
//
// Semantics follow the reference's portable codec
// (ccdl_comm/quantization/torch_fallback.py:24-36): fp32 arithmetic, IEEE
// division for absmax/127 and p/scale, round-half-even, eps clamp on the scale.
#include "quant_pack_block.h"

namespace lbc {
namespace {

using namespace quant;

template <typename XT, typename RT, typename DT, int G, int VEC, int MODE, int TILES>
__global__ __launch_bounds__(kBlock) void quant_pack_kernel(const QuantArgs a) {
    quant_pack_block<XT, RT, DT, G, VEC, MODE, TILES>(a, blockIdx.x, gridDim.x, blockIdx.y);
}

template <typename XT, typename RT, typename DT, int G, int VEC, int TILES>
hipError_t launch_tiles(int mode, const QuantArgs &a, int world, hipStream_t stream) {
    using T = quant_tiling<VEC, TILES>;
    const int64_t groups = (a.shard_numel + G - 1) / G;
    const int64_t padded = groups * G;
    const int64_t blocks = (padded + T::BLOCK_ELEMS - 1) / T::BLOCK_ELEMS;
    if (blocks == 0 || world == 0) return hipSuccess;
    if (blocks > 0x7FFFFFFFLL || world > 65535) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(world));
    // A single payload without a residual keeps its codes within reach of the launch that reads them next: plain stores up to
    // 4 Mi fp32 elements and written through beyond; 16-bit tensors plain beyond 20 Mi elements.  us of quantize + decode, codes
    // non-temporal / plain / written through, three tensors in rotation and (in brackets) enough of them to outrun the
    // last-level cache: fp32 4.1 M 8.9 / 9.3 / 8.6 (10.9 / 9.7 / -), 5.2 M 12.7 / 11.8 / 11.2 (12.6 / 11.1 / 11.5), 6.6 M
    // 14.9 / 16.0 / 14.3 (14.7 / 13.4 / 13.6), 13.1 M 26.5 / 26.2 / 23.9 (25.1 / 22.9 / 22.6), 26.2 M 46.3 / 41.5 / 42.3 (45.5 /
    // 41.2 / 41.2); with the reduce of two payloads as the reader 13.1 M 28.2 / 27.6 / 26.2 (27.2 / 25.6 / 26.0); of four and eight
    // within 2 % either way, but 4.3 and 5.2 M 3 % slower (4 payloads in rotation 13.2 / 13.7 / 13.7 and 15.2 / 15.6 / 15.6).
    // 16-bit, non-temporal / plain, decode and reduce of two, four and eight payloads: 8.4 M 10.0 / 10.0, 14.4 / 16.3, 17.2 /
    // 16.8, 22.6 / 22.4 (13.5 / 11.9, 15.0 / 14.7, 18.0 / 17.6, 22.7 / 22.5), 13.1 M 13.3 / 13.3, 19.9 / 22.0, 22.9 / 23.1,
    // 31.6 / 30.8 (17.9 / 15.5, 20.6 / 19.3, 23.9 / 22.9, 32.7 / 31.3), 19.7 M 18.8 / 18.4, 26.7 / 26.7, 32.2 / 31.2, 46.4 / 44.9,
    // 26.2 M 25.0 / 24.8, 32.7 / 32.2, 39.8 / 39.2, 58.9 / 55.8 (30.5 / 27.0, 34.9 / 32.6, 40.7 / 39.4, 60.3 / 57.1): below the
    // line few buckets of two ranks lose up to 18 %; written through, the decode loses up to 15 % up to 23 M.
    // A launch with outputs of its own (the first one with error feedback, which has no residual yet) is not what the codes wait
    // for: it keeps the hint up to 10 Mi elements of four a lane and writes through beyond.  us of the launch with an fp32 new
    // residual, non-temporal / plain / written through, in rotation (beyond the cache): fp32 3.0 M 5.5 / 5.9 / 6.1 (5.9 / 6.2 /
    // 6.4), 5.2 M 7.9 / 8.4 / 8.8 (9.0 / 9.2 / 9.6), 9.5 M 15.3 / 15.7 / 15.2 (15.9 / 15.8 / 15.5), 26.2 M 39.2 / 37.3 / 37.0; bf16
    // 4.3 M 8.0 / 8.9 / 9.1 (8.3 / 9.0 / 8.8), 8.4 M 12.4 / 13.3 / 13.0 (12.8 / 13.4 / 13.1), 11 M 14.7 / 15.0 / 14.6, 26.2 M
    // 31.5 / 30.1 / 29.7.
    if constexpr (is_void_t<RT>::value) {
        const bool outputs = a.new_residual != nullptr || a.restored != nullptr || a.prepared != nullptr;
        const bool whole = mode == kStream && world == 1;
        if constexpr (VEC == 4 && TILES > 1) {
            if (whole && a.numel > int64_t{outputs ? 10 : 4} << 20) {
                hipLaunchKernelGGL((quant_pack_kernel<XT, RT, DT, G, VEC, kStreamThrough, TILES>), grid, dim3(kBlock), 0, stream, a);
                return hipGetLastError();
            }
        }
        if constexpr (VEC == 8 ? TILES > 1 : sizeof(XT) == 4) {   // four 16-bit elements a lane: always with outputs
            if (whole && (VEC == 8 ? a.numel > int64_t{20} << 20 : !outputs)) {
                hipLaunchKernelGGL((quant_pack_kernel<XT, RT, DT, G, VEC, kStreamKept, TILES>), grid, dim3(kBlock), 0, stream, a);
                return hipGetLastError();
            }
        }
    }
    switch (mode) {
        case kStream: hipLaunchKernelGGL((quant_pack_kernel<XT, RT, DT, G, VEC, kStream, TILES>), grid, dim3(kBlock), 0, stream, a); break;
        case kVector: hipLaunchKernelGGL((quant_pack_kernel<XT, RT, DT, G, VEC, kVector, TILES>), grid, dim3(kBlock), 0, stream, a); break;
        default: hipLaunchKernelGGL((quant_pack_kernel<XT, RT, DT, G, VEC, kUnaligned, TILES>), grid, dim3(kBlock), 0, stream, a); break;
    }
    return hipGetLastError();
}

// One tile a wavefront while the tiles fit the chip's wavefront slots (2 Mi elements of four a lane, 4 Mi of eight):
// one tile against the usual number, us: fp32 10,007 elements 1.9 / 2.3, 65,536 2.1 / 2.4, 1 Mi 2.9 / 3.2, 2 Mi 3.6 / 3.9,
// 4 Mi 5.7 / 5.5, 6.6 M 8.9 / 7.4; bf16 10,007 2.0 / 2.2, 1 Mi 2.6 / 2.8, 4 Mi 3.8 / 3.9, 13.1 M 9.5 / 8.9; bf16 with an
// fp32 residual 10,007 2.3 / 3.5, 1 Mi 4.2 / 4.5, 2 Mi 6.0 / 6.3, 6.6 M 15.0 / 14.0.
template <typename XT, typename RT, typename DT, int G, int VEC>
hipError_t launch_typed(int mode, const QuantArgs &a, int world, hipStream_t stream) {
    if (a.numel <= kResidentWaves * kWave * VEC) return launch_tiles<XT, RT, DT, G, VEC, 1>(mode, a, world, stream);
    return launch_tiles<XT, RT, DT, G, VEC, quant_unroll<VEC>()>(mode, a, world, stream);
}

template <typename XT, typename RT, typename DT, int VEC>
hipError_t launch_group(int g, int mode, const QuantArgs &a, int world, hipStream_t s) {
    switch (g) {
        case 64: return launch_typed<XT, RT, DT, 64, VEC>(mode, a, world, s);
        case 32: return launch_typed<XT, RT, DT, 32, VEC>(mode, a, world, s);
        case 16: return launch_typed<XT, RT, DT, 16, VEC>(mode, a, world, s);
        default: return hipErrorNotSupported;
    }
}

// residual type in {none, float, XT}; restored type in {float, XT}.  Pure 16-bit
// calls take 8 elements per lane, everything touching an fp32 tensor takes 4.
template <typename XT>
hipError_t launch_x(int x_dtype, int r_dtype, int d_dtype, bool outputs, int g, int mode, const QuantArgs &a,
                    int world, hipStream_t s) {
    constexpr int WIDE = 16 / sizeof(XT);
    const bool d_is_x = d_dtype == x_dtype;
    if (!d_is_x && d_dtype != kF32) return hipErrorNotSupported;
    if (r_dtype == kNone) {
        if (!outputs || d_is_x) return launch_group<XT, void, XT, WIDE>(g, mode, a, world, s);
        return launch_group<XT, void, float, 4>(g, mode, a, world, s);
    }
    if (r_dtype == x_dtype) {
        // Without `restored` and `new_residual` nothing is rounded to DT, so the call is as narrow as its tensors:
        // 13.1 M bf16 elements with a bf16 residual and their sum as a second output (the all_gather hook's quantize)
        // take the same 16.5 us either way, 1.3 M 4.4 us with 8 elements a lane and 4.6 us with 4, 131,072 2.9 and 3.1 us.
        if (d_is_x || !outputs) return launch_group<XT, XT, XT, WIDE>(g, mode, a, world, s);
        return launch_group<XT, XT, float, 4>(g, mode, a, world, s);
    }
    if (r_dtype == kF32) {
        if (d_is_x) return launch_group<XT, float, XT, 4>(g, mode, a, world, s);
        return launch_group<XT, float, float, 4>(g, mode, a, world, s);
    }
    return hipErrorNotSupported;
}

}  // namespace

int quant_pack_vec(int x_dtype, int r_dtype, int d_dtype, bool outputs) {
    if (x_dtype == kF32) return 4;
    const bool d_is_x = d_dtype == x_dtype;
    if (r_dtype == kNone) return (!outputs || d_is_x) ? 8 : 4;
    if (r_dtype == x_dtype) return (d_is_x || !outputs) ? 8 : 4;
    return 4;
}

hipError_t launch_quant_pack(int x_dtype, int r_dtype, int d_dtype, bool outputs, int group_size, int mode,
                             const QuantArgs &args, int world, hipStream_t stream) {
    switch (x_dtype) {
        case kF32: return launch_x<float>(x_dtype, r_dtype, d_dtype, outputs, group_size, mode, args, world, stream);
        case kF16: return launch_x<f16>(x_dtype, r_dtype, d_dtype, outputs, group_size, mode, args, world, stream);
        case kBF16: return launch_x<bf16>(x_dtype, r_dtype, d_dtype, outputs, group_size, mode, args, world, stream);
        default: return hipErrorNotSupported;
    }
}

}  // namespace lbc
