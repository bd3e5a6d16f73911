// Sums over the lanes of a wave, shared by the sweeps for many channels (sig_rows.hip, sig_rows_mfma.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "sig_kernels.h"

namespace sigamd {

template <int CTRL>
__device__ __forceinline__ float dpp_moved(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_moved(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float lane_value(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ __forceinline__ double lane_value(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
}
// every lane receives the sum over its row of 16 lanes
template <typename T>
__device__ __forceinline__ T row_sum_rows(T v)
{
    v += dpp_moved<0xB1>(v);        // quad_perm [1, 0, 3, 2]
    v += dpp_moved<0x4E>(v);        // quad_perm [2, 3, 0, 1]
    v += dpp_moved<0x141>(v);       // row_half_mirror
    v += dpp_moved<0x140>(v);       // row_mirror
    return v;
}
// sum over the 64 lanes, valid in every lane
template <typename T>
__device__ __forceinline__ T wave_sum_rows(T v)
{
    v = row_sum_rows(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}
// lanes 0-31: lo[lane] + lo[lane + 32];  lanes 32-63: hi[lane - 32] + hi[lane]
__device__ __forceinline__ float half_sums(float lo, float hi)
{
    const auto r = __builtin_amdgcn_permlane32_swap(unsigned(__float_as_int(lo)), unsigned(__float_as_int(hi)), false, false);
    return __int_as_float(int(r[0])) + __int_as_float(int(r[1]));
}
__device__ __forceinline__ double half_sums(double lo, double hi) { return pair_sum32(lo, hi); }
// rows of 16 lanes:  0: a0 + a1,  1: b0 + b1,  2: a2 + a3,  3: b2 + b3   (ai, bi: row i of a, b)
__device__ __forceinline__ float quarter_sums(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(unsigned(__float_as_int(a)), unsigned(__float_as_int(b)), false, false);
    return __int_as_float(int(r[0])) + __int_as_float(int(r[1]));
}
// the sums of two values over the 64 lanes for the price of one and a half: the half-waves first exchange halves
template <typename T>
__device__ __forceinline__ void wave_sum_two(T a, T b, T& sum_a, T& sum_b)
{
    const T v = row_sum_rows(half_sums(a, b));
    sum_a = lane_value(v, 0) + lane_value(v, 16);
    sum_b = lane_value(v, 32) + lane_value(v, 48);
}

}  // namespace sigamd
