// Wavefront (64-lane) primitives for gfx950: reductions, segmented scans and
// lane masks built on ds_bpermute / DPP-backed shuffles.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace sgipc {

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// orders a wave's LDS writes before its lanes' later reads
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Reductions over the wave without the LDS pipe: lane halves and rows meet by
// the permlane swaps, lanes of a row by DPP rotations.  A rotation by d stands
// for lane ^ d: by then the values of a row repeat every 2 d lanes.  The sums
// therefore pair the same lanes in the same order as six __shfl_xor steps (bit
// for bit), without their six round trips through LDS: with 6 to 9 block sums per
// PCG iteration, all of them latency, the FP64 solve of a 16^3 grid takes 2.79
// instead of 3.16 ms, one MAS apply 60 instead of 68 us.  The whole wave has to
// be active.
template <int kCtrl, typename T>
__device__ __forceinline__ T dpp_row(T v)
{
    constexpr int kWords = sizeof(T) / 4;
    int w[kWords];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int k = 0; k < kWords; ++k) w[k] = __builtin_amdgcn_update_dpp(0, w[k], kCtrl, 0xF, 0xF, true);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// a, b: the values of the two halves (kHalf = 32) or of a row pair (16)
template <int kHalf, typename T>
__device__ __forceinline__ void swap_halves(T v, T& a, T& b)
{
    constexpr int kWords = sizeof(T) / 4;
    unsigned w[kWords], x[kWords], y[kWords];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int k = 0; k < kWords; ++k) {
        auto r = kHalf == 32 ? __builtin_amdgcn_permlane32_swap(w[k], w[k], false, false)
                             : __builtin_amdgcn_permlane16_swap(w[k], w[k], false, false);
        x[k] = r[0];
        y[k] = r[1];
    }
    __builtin_memcpy(&a, x, sizeof(T));
    __builtin_memcpy(&b, y, sizeof(T));
}

template <typename T, typename F>
__device__ __forceinline__ T wave_reduce(T v, F f)
{
    static_assert(sizeof(T) % 4 == 0, "whole 32-bit words");
    T a, b;
    swap_halves<32>(v, a, b);
    v = f(a, b);
    swap_halves<16>(v, a, b);
    v = f(a, b);
    v = f(v, dpp_row<0x128>(v));  // row_ror:8
    v = f(v, dpp_row<0x124>(v));
    v = f(v, dpp_row<0x122>(v));
    return f(v, dpp_row<0x121>(v));
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
    return wave_reduce(v, [](T x, T y) { return x + y; });
}

template <typename T>
__device__ __forceinline__ T wave_max(T v)
{
    return wave_reduce(v, [](T x, T y) { return y > x ? y : x; });
}

// Sum over the aligned group of W lanes, in all of them (every lane of the
// group active), in the order of the __shfl_xor steps from W / 2 down to 1.
template <int W, typename T>
__device__ __forceinline__ T group_sum(T v)
{
    static_assert(W == 8 || W == 16 || W == 32, "half a row, a row, a row pair");
    if constexpr (W == 8) {
        v += dpp_row<0x1B>(dpp_row<0x141>(v));  // row_half_mirror, quad_perm [3,2,1,0]: lane ^ 4
        v += dpp_row<0x4E>(v);                  // quad_perm: lane ^ 2
        return v + dpp_row<0xB1>(v);
    } else {
        if constexpr (W == 32) {
            T a, b;
            swap_halves<16>(v, a, b);
            v = a + b;
        }
        v += dpp_row<0x128>(v);  // row_ror:8
        v += dpp_row<0x124>(v);
        v += dpp_row<0x122>(v);
        return v + dpp_row<0x121>(v);
    }
}

// Sums of three values by key within aligned groups of W lanes, all groups of
// the wave at a time: write(key, s0, s1, s2) runs once per distinct key >= 0
// of a group, as many rounds as the group with the most keys has.
template <int W, typename T, typename F>
__device__ __forceinline__ void group_key_sums(int key, T v0, T v1, T v2, F write)
{
    const int lane = threadIdx.x & 63, base = lane & ~(W - 1);
    bool pending = key >= 0;
    while (true) {
        const uint64_t act = __ballot(pending);
        if (act == 0) break;
        const uint32_t mask = (uint32_t)(act >> base) & (uint32_t)((1ull << W) - 1);
        const int leader = mask != 0 ? base + __ffs(mask) - 1 : lane;
        const int k = __shfl(key, leader, 64);
        const bool mine = pending && key == k;
        const T s0 = group_sum<W>(mine ? v0 : T(0));
        const T s1 = group_sum<W>(mine ? v1 : T(0));
        const T s2 = group_sum<W>(mine ? v2 : T(0));
        if (mine && lane == leader) write(k, s0, s1, s2);
        if (mine) pending = false;
    }
}

// Workgroup b of n -> its place in a contiguous run per XCD: the 8 XCDs take
// workgroups in turn, so XCD b % 8 gets run [x n / 8 ..) and its L2 holds what
// neighbours share.  A bijection on [0, n).
__device__ __forceinline__ int xcd_run(int b, int n)
{
    const int x = b & 7, q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// Index of the highest set bit of m that is <= lane (m must have one such bit).
__device__ __forceinline__ int seg_start_from_heads(uint64_t heads, int lane)
{
    uint64_t upto = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
    return 63 - __clzll(heads & upto);
}

// Inclusive segmented prefix sum across the wave: after the call the last lane
// of every segment holds the segment total.  `start` is the first lane of the
// caller's segment.
template <typename T>
__device__ __forceinline__ T seg_inclusive_sum(T v, int lane, int start)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        T t = __shfl_up(v, off, 64);
        if (lane - off >= start) v += t;
    }
    return v;
}

// Block-wide deterministic sum of `v` (blockDim.x a multiple of 64, <= 1024).
// Every wave adds the waves' sums itself, so one barrier publishes them and
// one frees smem for the next use.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T* smem /* >= 16 */)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63;
    if (lane == 0) smem[threadIdx.x >> 6] = v;
    __syncthreads();
    const int nw = blockDim.x >> 6;
    const T s = wave_sum(lane < nw ? smem[lane] : T(0));
    __syncthreads();
    return s;
}

// Deterministic sum of n partials by a whole workgroup (fixed order).
__device__ __forceinline__ double block_sum_array(const double* __restrict__ a, int n, double* smem)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += a[i];
    return block_sum(s, smem);
}

__device__ __forceinline__ void atomic_add(double* p, double v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void atomic_add(float* p, float v) { unsafeAtomicAdd(p, v); }

}  // namespace sgipc
