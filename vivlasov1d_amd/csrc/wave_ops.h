// Wavefront-wide sums and neighbour exchange by DPP (data moved between the
// lanes' registers: a few cycles a step, where a shuffle goes through the LDS
// unit, ~100 cycles for a double).  All 64 lanes must be active.
#pragma once

#include <hip/hip_runtime.h>

namespace vv {
namespace {

// DPP controls: lane i takes lane i -/+ n of its row of 16 (0 past the row);
// lane 15 of each row to the next row; lane 31 to rows 2 and 3
constexpr int kDppShr = 0x110, kDppShl = 0x100, kDppBcast15 = 0x142, kDppBcast31 = 0x143;

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROWS, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_move(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xf, true));
}

__device__ __forceinline__ double read_lane(double x, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}
__device__ __forceinline__ float read_lane(float x, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// sum over the wavefront, in every lane (fixed tree: prefix sums of each row of
// 16 by 1, 2, 4, 8, then the rows)
__device__ __forceinline__ double wave_sum(double v)
{
    v += dpp_move<kDppShr + 1, 0xf>(v);
    v += dpp_move<kDppShr + 2, 0xf>(v);
    v += dpp_move<kDppShr + 4, 0xf>(v);
    v += dpp_move<kDppShr + 8, 0xf>(v);
    v += dpp_move<kDppBcast15, 0xa>(v);
    v += dpp_move<kDppBcast31, 0xc>(v);
    return read_lane(v, 63);
}

}  // namespace
}  // namespace vv
