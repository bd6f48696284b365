// sort_scan.h -- workgroup sorts, prefix sums and lists of patches of the setup kernels.
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

// The patches (of ps elements, by the elements' positions epos) that hold the node
// of the calling thread, with the incidences inc[b0..b1): *total their number, *rank
// how many come before patch p.  All NT threads call it; those whose node lies in
// one patch only, or that have none, with shared = false (0 and -1 then).  A thread
// lists its node's patches one after the other, a pass over the incidences for
// each, up to kManyInc incidences; a node of more is done by the whole workgroup,
// which marks its patches in a set of kPatchWindow bits (one after the other in
// one thread, a node of 9,800 Tet4 in 21 patches took 74 ms).
constexpr int kManyInc = 48, kPatchWindow = 32768;
template <int NT>
__device__ __forceinline__ void patches_of_node(bool shared, int b0, int b1, int npe, int ps, int npatch, int p,
                                                const int32_t *__restrict__ inc, const int32_t *__restrict__ epos, int *total,
                                                int *rank) {
    __shared__ uint32_t set[kPatchWindow / 32];
    __shared__ int who[NT];
    const int t = threadIdx.x;
    const bool many = shared && b1 - b0 > kManyInc;
    *total = 0;
    *rank = shared ? 0 : -1;
    if (shared && !many)
        for (int last = -1;;) {
            int next = INT32_MAX;
            for (int k = b0; k < b1; ++k) {
                const int o = epos[inc[k] / npe] / ps;
                if (o > last && o < next) next = o;
            }
            if (next == INT32_MAX) break;
            ++*total;
            *rank += next < p;
            last = next;
        }
    if (!__syncthreads_or(many)) return;
    int n;
    const int at = block_scan<NT>(many, &n);
    if (many) who[at] = t;
    __shared__ int lo, hi;
    for (int j = 0; j < n; ++j) {
        __syncthreads();
        if (t == who[j]) {
            lo = b0;
            hi = b1;
        }
        __syncthreads();
        const int k0 = lo, k1 = hi;
        int all = 0, before = 0;
        for (int w0 = 0; w0 < npatch; w0 += kPatchWindow) {
            const int words = (min(kPatchWindow, npatch - w0) + 31) / 32;
            for (int i = t; i < words; i += NT) set[i] = 0;
            __syncthreads();
            for (int k = k0 + t; k < k1; k += NT) {
                const int o = epos[inc[k] / npe] / ps - w0;
                if (o >= 0 && o < kPatchWindow) atomicOr(&set[o >> 5], 1u << (o & 31));
            }
            __syncthreads();
            int a = 0, b = 0, sum;
            for (int i = t; i < words; i += NT) {
                const int first = w0 + 32 * i;  // the bits of patches below p
                const uint32_t below = p - first >= 32 ? ~0u : (p <= first ? 0u : (1u << (p - first)) - 1u);
                a += __popc(set[i]);
                b += __popc(set[i] & below);
            }
            (void)block_scan<NT>(a, &sum);
            all += sum;
            (void)block_scan<NT>(b, &sum);
            before += sum;
        }
        if (t == who[j]) {
            *total = all;
            *rank = before;
        }
    }
}

}  // namespace jfem
