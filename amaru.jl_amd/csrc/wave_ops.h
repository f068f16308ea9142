// Sums over a 64-lane wave by DPP moves.
#pragma once
#include <hip/hip_runtime.h>

// v of the lane that DPP control CTRL pairs with this one
template <int CTRL>
__device__ inline double dpp_pair(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

__device__ inline double read_lane(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the wave by one fixed tree, the same value in every lane: pairs,
// quads, eights and rows of 16 by DPP moves (a register move each, where a
// shuffle is an LDS round trip), then the four rows.
__device__ inline double wave_sum(double v)
{
    v += dpp_pair<0xB1>(v);   // quad_perm 1,0,3,2
    v += dpp_pair<0x4E>(v);   // quad_perm 2,3,0,1
    v += dpp_pair<0x141>(v);  // row_half_mirror
    v += dpp_pair<0x140>(v);  // row_mirror
    return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}
