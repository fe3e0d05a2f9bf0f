// wave_device.h -- sums over a wave by data-parallel moves, without LDS.
#pragma once

#include <hip/hip_runtime.h>

namespace dmed {

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v)
{
    // lanes without a source, or in rows outside ROWS, add 0
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sum over the wave, valid in lane 63: shifts by 1, 2, 4, 8 inside the rows
// of 16 lanes, then row 0 into 1 and 2 into 3, then rows 0-1 into 2-3
__device__ __forceinline__ double wave_sum63(double v)
{
    v = dpp_add<0x111, 0xf>(v);
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);
    v = dpp_add<0x143, 0xc>(v);
    return v;
}

}  // namespace dmed
