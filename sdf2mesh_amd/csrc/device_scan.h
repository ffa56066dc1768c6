// device_scan.h - prefix sums over the lanes of a wave with data-parallel moves (a register
// operand shifted by lanes: a few cycles, against some 130 for a shuffle through LDS).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace s2m {

// Inclusive prefix sum within each row of 16 lanes.
__device__ __forceinline__ uint32_t row_scan(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
    return x;
}

// Inclusive prefix sum over the 64 lanes (the rows' totals passed on; all lanes active).
__device__ __forceinline__ uint32_t wave_scan(uint32_t x)
{
    x = row_scan(x);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

// The same for another operation on floats, `none` its neutral element.
template <class Op>
__device__ __forceinline__ float wave_scan(float x, float none, const Op& op)
{
    const int o = (int)__float_as_uint(none);
    auto from = [&](auto move) { return __uint_as_float((uint32_t)move(o, (int)__float_as_uint(x))); };
    x = op(x, from([](int n, int v) { return __builtin_amdgcn_update_dpp(n, v, 0x111, 0xf, 0xf, false); }));
    x = op(x, from([](int n, int v) { return __builtin_amdgcn_update_dpp(n, v, 0x112, 0xf, 0xf, false); }));
    x = op(x, from([](int n, int v) { return __builtin_amdgcn_update_dpp(n, v, 0x114, 0xf, 0xf, false); }));
    x = op(x, from([](int n, int v) { return __builtin_amdgcn_update_dpp(n, v, 0x118, 0xf, 0xf, false); }));
    x = op(x, from([](int n, int v) { return __builtin_amdgcn_update_dpp(n, v, 0x142, 0xa, 0xf, false); }));
    x = op(x, from([](int n, int v) { return __builtin_amdgcn_update_dpp(n, v, 0x143, 0xc, 0xf, false); }));
    return x;
}
__device__ __forceinline__ float wave_min(float x, float none) { return wave_scan(x, none, [](float a, float b) { return fminf(a, b); }); }
__device__ __forceinline__ float wave_max(float x, float none) { return wave_scan(x, none, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ float wave_sum(float x) { return wave_scan(x, 0.0f, [](float a, float b) { return a + b; }); }

// The last lane's value, and the value of the lane below (`none` for lane 0).
__device__ __forceinline__ float last_lane(float x)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), 63));
}
__device__ __forceinline__ float lane_below(float x, float none)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(none), (int)__float_as_uint(x), 0x138,
                                                                 0xf, 0xf, false));  // wave_shr:1
}

}  // namespace s2m
