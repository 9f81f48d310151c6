// Sums and products over one wave (gfx950), shared by the small dense kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace qm {

// v of the lane R places on inside a row of 16 (rotation), through DPP
template <int R>
__device__ __forceinline__ double row_ror(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x120 + R, 0xf, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x120 + R, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v of lane `lane` (uniform), as a scalar
__device__ __forceinline__ double lane_value(double v, int lane) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum over the wave, the same bits in every lane: rows of 16 by DPP rotations,
// the four rows' sums through scalar registers.  No LDS: an exchange through
// ds_bpermute takes ~130 cycles, and six of them follow one another in a
// butterfly sum.
__device__ __forceinline__ double wave_sum(double v) {
    v += row_ror<1>(v);
    v += row_ror<2>(v);
    v += row_ror<4>(v);
    v += row_ror<8>(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

__device__ __forceinline__ double wave_prod(double v) {
    v *= row_ror<1>(v);
    v *= row_ror<2>(v);
    v *= row_ror<4>(v);
    v *= row_ror<8>(v);
    return (lane_value(v, 0) * lane_value(v, 16)) * (lane_value(v, 32) * lane_value(v, 48));
}

}  // namespace qm
