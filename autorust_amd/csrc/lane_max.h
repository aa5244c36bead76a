// Maxima and sums over groups of lanes without LDS: a __shfl_xor is an LDS round trip of some 100 cycles, and a reduction is a chain of
// them; the vector ALU's own lane exchanges take a few cycles each.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace arhip {

// x of the lane that CTRL names
template <int CTRL>
__device__ __forceinline__ float dpp_read(float x)
{
    const int u = __float_as_int(x);
    return __int_as_float(__builtin_amdgcn_update_dpp(u, u, CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ float dpp_max(float x) { return fmaxf(x, dpp_read<CTRL>(x)); }

// largest x of each aligned group of G lanes (8, 16, 32 or 64), in every lane of it
template <int G>
__device__ __forceinline__ float lane_group_max(float x)
{
    static_assert(G == 8 || G == 16 || G == 32 || G == 64, "group of lanes");
    x = dpp_max<0xB1>(x);                    // quad_perm [1,0,3,2]: lane ^ 1
    x = dpp_max<0x4E>(x);                    // quad_perm [2,3,0,1]: lane ^ 2
    x = dpp_max<0x141>(x);                   // row_half_mirror: the other four of eight
    if constexpr (G >= 16) x = dpp_max<0x140>(x);  // row_mirror: the other eight of sixteen
    if constexpr (G >= 32) {
        const uint32_t u = __float_as_uint(x);
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    if constexpr (G == 64) {
        const uint32_t u = __float_as_uint(x);
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    return x;
}

// x, the same in every lane, as a scalar
__device__ __forceinline__ float wave_value(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }

// sum of x over the 64 lanes, in every lane
__device__ __forceinline__ float xrow_max(float x)  // of lane and lane ^ 16
{
    const uint32_t u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float lane_sum_16(float x)  // of each aligned group of 16, in every lane of it
{
    x += dpp_read<0xB1>(x);
    x += dpp_read<0x4E>(x);
    x += dpp_read<0x141>(x);
    return x + dpp_read<0x140>(x);
}
__device__ __forceinline__ float lane_sum(float x)
{
    x = lane_sum_16(x);
    uint32_t u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    u = __float_as_uint(x);
    const auto t = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}

}  // namespace arhip
