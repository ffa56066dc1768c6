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

}  // namespace s2m
