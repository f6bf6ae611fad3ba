// Helpers of the kernels whose work-group carries a tile of 32 rows through several products (16 lanes a row).
#pragma once

#include "common.h"

namespace bnb {

// Waits for this wave's LDS traffic only: operands requested from memory stay on their way across the barrier.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v)
{
    return v + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), CTRL, 0xf, 0xf, false));
}
// Sum over the 16 lanes of a row, in all of them.
__device__ __forceinline__ float sum16(float v)
{
    v = dpp_add<0x128>(v);  // row_ror:8, 4, 2, 1
    v = dpp_add<0x124>(v);
    v = dpp_add<0x122>(v);
    return dpp_add<0x121>(v);
}

}  // namespace bnb
