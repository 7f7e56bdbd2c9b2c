// Per-workgroup sums of 3-vectors by vertex, for gradient scatters: elements
// next to each other share vertices, and an FP64 atomic in LDS is far cheaper
// than one in memory.  A hash table in LDS takes the additions; the distinct
// vertices are then added to memory once per workgroup.  A vertex that finds
// no slot within kProbes goes to memory directly.
#pragma once
#include "wave_ops.hpp"

namespace sgipc {

template <int N>  // slots, a power of two
struct VertexSums {
    static constexpr int kProbes = 8;
    int key[N];
    double sum[3][N];

    // all threads; a barrier follows
    __device__ __forceinline__ void init()
    {
        for (int i = threadIdx.x; i < N; i += blockDim.x) {
            key[i] = -1;
            sum[0][i] = sum[1][i] = sum[2][i] = 0.0;
        }
        __syncthreads();
    }
    __device__ __forceinline__ void add(int v, double x, double y, double z, double* __restrict__ grad)
    {
        unsigned h = ((unsigned)v * 2654435761u) >> (32 - __builtin_ctz(N));
        for (int t = 0; t < kProbes; ++t, h = (h + 1) & (N - 1)) {
            const int k = atomicCAS(&key[h], -1, v);
            if (k == -1 || k == v) {
                atomicAdd(&sum[0][h], x);
                atomicAdd(&sum[1][h], y);
                atomicAdd(&sum[2][h], z);
                return;
            }
        }
        atomic_add(grad + 3L * v, x);
        atomic_add(grad + 3L * v + 1, y);
        atomic_add(grad + 3L * v + 2, z);
    }
    // all threads; consecutive threads take the components of one vertex
    __device__ __forceinline__ void flush(double* __restrict__ grad)
    {
        __syncthreads();
        for (int i = threadIdx.x; i < 3 * N; i += blockDim.x) {
            const int h = i / 3, c = i % 3, v = key[h];
            if (v >= 0) atomic_add(grad + 3L * v + c, sum[c][h]);
        }
    }
};

}  // namespace sgipc
