// sort_scan.h -- workgroup sorts and prefix sums of the setup kernels.
#pragma once

#include "jfem_device.h"

namespace jfem {

// Exclusive scan over the workgroup's NT threads; *total: the sum, to every thread.
template <int NT> __device__ __forceinline__ int block_scan(int v, int *total) {
    __shared__ int ws[NT / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int s = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(s, off, 64);
        if (lane >= off) s += u;
    }
    if (lane == 63) ws[wid] = s;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        if (w < wid) before += ws[w];
        all += ws[w];
    }
    __syncthreads();
    *total = all;
    return before + s - v;
}

// Ascending order (bitonic) of the n (a power of two) keys in LDS, NT threads.
template <int NT, typename K> __device__ __forceinline__ void sort_keys(K *key, int n) {
    for (int size = 2; size <= n; size <<= 1)
        for (int s = size >> 1; s > 0; s >>= 1) {
            __syncthreads();
            for (int q = (int)threadIdx.x; q < n / 2; q += NT) {
                const int i = 2 * q - (q & (s - 1)), j = i + s;
                const K u = key[i], v = key[j];
                if ((u > v) == ((i & size) == 0)) {
                    key[i] = v;
                    key[j] = u;
                }
            }
        }
    __syncthreads();
}

}  // namespace jfem
