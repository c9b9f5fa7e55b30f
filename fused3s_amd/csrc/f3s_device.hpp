// f3s_device.hpp -- device-side building blocks (wave64, gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace f3s {

constexpr int kWave = 64;

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// Workgroup barrier that orders LDS only.  __syncthreads() also fences
// global memory, which makes every wave wait for all of its outstanding
// vector-memory loads (s_waitcnt vmcnt(0)) at each barrier; this one waits
// for LDS operations only, so loads issued ahead of time stay in flight.
// Global stores made before it are NOT visible to the other waves after it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Orders this wave's LDS accesses between its lanes.  The LDS unit runs a
// wave's operations in their order, so only the compiler has to be held.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// Inclusive scan over the 64 lanes of a wave.
template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v)
{
    const int lane = lane_id();
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        T o = __shfl_up(v, off, kWave);
        if (lane >= off) v += o;
    }
    return v;
}

// Inclusive prefix sum over the wave with DPP row shifts and row broadcasts.
__device__ __forceinline__ int wave_scan_incl(int x)
{
    int s = x;
    s += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
    s += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
    s += __builtin_amdgcn_update_dpp(0, x, 0x113, 0xf, 0xf, true);   // row_shr:3
    s += __builtin_amdgcn_update_dpp(0, s, 0x114, 0xf, 0xe, true);   // row_shr:4, lanes 4-15
    s += __builtin_amdgcn_update_dpp(0, s, 0x118, 0xf, 0xc, true);   // row_shr:8, lanes 8-15
    s += __builtin_amdgcn_update_dpp(0, s, 0x142, 0xa, 0xf, true);   // row_bcast:15 -> rows 1, 3
    s += __builtin_amdgcn_update_dpp(0, s, 0x143, 0xc, 0xf, true);   // row_bcast:31 -> rows 2, 3
    return s;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Exclusive scan across a workgroup of NT threads (NT a multiple of 64);
// `total` receives the workgroup sum.  `lds` needs NT/64 elements.  Contains
// barriers: every thread of the workgroup must call it.
template <int NT, typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* lds, T& total)
{
    constexpr int NW = NT / kWave;
    const int lane = lane_id();
    const int wid = threadIdx.x / kWave;
    T inc = wave_inclusive_scan(v);
    if (lane == kWave - 1) lds[wid] = inc;
    __syncthreads();
    T base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        T s = lds[i];
        if (i < wid) base += s;
        tot += s;
    }
    __syncthreads();
    total = tot;
    return base + inc - v;
}

}  // namespace f3s
