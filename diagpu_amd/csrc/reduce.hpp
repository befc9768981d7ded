// Deterministic fp64 sums across a grid: every workgroup stores one partial
// with a plain store; a one-workgroup kernel launched after it adds the
// partials in index order.  The launch boundary makes the partials visible,
// so no device-scope fence is needed inside the producing kernel (on gfx950
// such a fence writes back and invalidates the XCD's L2 -- per workgroup,
// that cost more than the kernels themselves).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace diagpu {

// x plus the value a DPP move brings (0 where it brings none)
template <int Ctrl, int RowMask> __device__ __forceinline__ double dpp_add(double x)
{
    const uint64_t v = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, Ctrl, RowMask, 0xf,
                                                              false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), Ctrl,
                                                              RowMask, 0xf, false);
    return x + __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The wave's sum, in lane 63: within rows of 16 lanes, then across the rows
// (moves between registers, no round trip through LDS hardware per step).
__device__ __forceinline__ double wave_sum63(double x)
{
    x = dpp_add<0x111, 0xf>(x);   // row_shr:1
    x = dpp_add<0x112, 0xf>(x);   // row_shr:2
    x = dpp_add<0x114, 0xf>(x);   // row_shr:4
    x = dpp_add<0x118, 0xf>(x);   // row_shr:8
    x = dpp_add<0x142, 0xa>(x);   // row_bcast:15
    return dpp_add<0x143, 0xc>(x);   // row_bcast:31
}

// Sum of `s` over the calling workgroup (kBlockSize lanes, every lane
// calls).  The result is valid in every lane.
template <int kBlockSize>
__device__ __forceinline__ double block_sum(double s)
{
    __shared__ double wsum[kBlockSize / 64];
    s = wave_sum63(s);
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    __syncthreads();   // wsum may still be read by a previous call
    if (lane == 63) wsum[wave] = s;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBlockSize / 64; ++w) t += wsum[w];
    return t;
}

// Workgroup `part` stores the sum of its lanes' `s` into partials[part].
template <int kBlockSize>
__device__ __forceinline__ void store_partial(double s, int part, double* partials)
{
    const double t = block_sum<kBlockSize>(s);
    if (threadIdx.x == 0) partials[part] = t;
}

}  // namespace diagpu
