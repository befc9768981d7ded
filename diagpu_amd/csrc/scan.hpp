// Workgroup-wide prefix sums for 64-lane waves (device helpers).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace diagpu {

// `x` moved between lanes by a DPP control; lanes that get nothing keep `id`.
template <int Ctrl, int RowMask>
__device__ __forceinline__ int32_t dpp_move(int32_t x, int32_t id)
{
    return __builtin_amdgcn_update_dpp(id, x, Ctrl, RowMask, 0xf, false);
}
template <int Ctrl, int RowMask>
__device__ __forceinline__ int64_t dpp_move(int64_t x, int64_t id)
{
    const int32_t lo = dpp_move<Ctrl, RowMask>((int32_t)x, (int32_t)id);
    const int32_t hi = dpp_move<Ctrl, RowMask>((int32_t)(x >> 32), (int32_t)(id >> 32));
    return ((int64_t)hi << 32) | (uint32_t)lo;
}

// Inclusive scan under `op` (identity `id`) over the wave's lanes: within
// rows of 16 lanes, then across the rows.  Lane 63 holds the wave's result.
template <typename T, typename Op>
__device__ __forceinline__ T wave_scan_dpp(T v, T id, Op op)
{
    v = op(v, dpp_move<0x111, 0xf>(v, id));   // row_shr:1
    v = op(v, dpp_move<0x112, 0xf>(v, id));   // row_shr:2
    v = op(v, dpp_move<0x114, 0xf>(v, id));   // row_shr:4
    v = op(v, dpp_move<0x118, 0xf>(v, id));   // row_shr:8
    v = op(v, dpp_move<0x142, 0xa>(v, id));   // row_bcast:15
    return op(v, dpp_move<0x143, 0xc>(v, id));   // row_bcast:31
}

// Inclusive prefix sum across the 64 lanes of a wave.
template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const T o = __shfl_up(v, s, 64);
        if (lane >= s) v += o;
    }
    return v;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s, 64);
    return v;
}

// Exclusive prefix sum over a workgroup of BLOCK threads (BLOCK a multiple
// of 64, at most 1024).  `total` receives the workgroup sum.  `lds` must hold
// BLOCK / 64 values.  Contains barriers: every thread must call it.
template <typename T, int BLOCK>
__device__ __forceinline__ T block_exclusive_scan(T v, T& total, T* lds)
{
    constexpr int kWaves = BLOCK / 64;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const T incl = wave_inclusive_scan(v);
    if (lane == 63) lds[wave] = incl;
    __syncthreads();
    T before = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const T s = lds[w];
        before += (w < wave) ? s : T(0);
        sum += s;
    }
    __syncthreads();
    total = sum;
    return before + incl - v;
}

}  // namespace diagpu
