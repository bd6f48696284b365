// mesh_lists.hip -- the lists of an uploaded mesh, built on the device (gfx950).
//
// From the connectivity: each node's element incidences in ascending order, the
// sorted 3x3-block pattern of K, and per block the element blocks (e, i, j) that
// are summed into it, ascending, for the deterministic assembly.  A mesh of
// 12,810 Tet10 elements took 4.3 ms of host time for these (16 threads: sort and
// binary search per row) and 0.5 ms of copies; the kernels here take 0.12 ms.
//
// Nothing in them depends on the order in which threads run: atomics only count
// and place, and every list is then put in order by rank.
//
// Reference: the node -> element map of ext/JuliaFEMCUDAExt.jl:179-193.
#include <algorithm>

#include "sort_scan.h"

namespace jfem {

// ------------------------------------------------------------------- scan ---
// Exclusive prefix sums of int32: per-block sums of kScan values, their scan by
// one workgroup, and the blocks again with their offsets.
constexpr int kScan = 4 * kBlock;

__global__ __launch_bounds__(kBlock) void k_scan_sums(int n, const int32_t *__restrict__ in, int32_t *__restrict__ bsum) {
    const int64_t i0 = (int64_t)blockIdx.x * kScan + 4 * threadIdx.x;
    int v = 0, total;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (i0 + j < n) v += in[i0 + j];
    (void)block_scan<kBlock>(v, &total);
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_scan_carry(int nb, int32_t *__restrict__ bsum, int32_t *__restrict__ last) {
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += 1024) {
        const int b = b0 + (int)threadIdx.x, v = b < nb ? bsum[b] : 0;
        int total;
        const int ex = block_scan<1024>(v, &total);
        if (b < nb) bsum[b] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) *last = carry;
}

__global__ __launch_bounds__(kBlock) void k_scan_add(int n, const int32_t *__restrict__ in, const int32_t *__restrict__ bsum,
                                                    int32_t *__restrict__ out) {
    const int64_t i0 = (int64_t)blockIdx.x * kScan + 4 * threadIdx.x;
    int v[4], s = 0, total;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = i0 + j < n ? in[i0 + j] : 0;
        s += v[j];
    }
    int o = bsum[blockIdx.x] + block_scan<kBlock>(s, &total);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (i0 + j < n) out[i0 + j] = o;
        o += v[j];
    }
}

// out[0..n]: the exclusive sums of in[0..n) and the total
static void scan(hipStream_t s, int n, const int32_t *in, int32_t *out, int32_t *bsum) {
    const int nb = (n + kScan - 1) / kScan;
    k_scan_sums<<<nb, kBlock, 0, s>>>(n, in, bsum);
    k_scan_carry<<<1, 1024, 0, s>>>(nb, bsum, out + n);
    k_scan_add<<<nb, kBlock, 0, s>>>(n, in, bsum, out);
}

// -------------------------------------------------------------- incidences ---
// One thread per incidence q = (e, i): the connectivity by local node, and the
// nodes' valences.
template <int NPE>
__global__ __launch_bounds__(kBlock) void k_conn_split(int n_el, const int32_t *__restrict__ connE, int32_t *__restrict__ conn,
                                                      int32_t *__restrict__ cnt) {
    const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (q >= (int64_t)n_el * NPE) return;
    const int a = connE[q];
    conn[(q % NPE) * n_el + q / NPE] = a;
    atomicAdd(&cnt[a], 1);
}

// Places the incidences in their nodes' ranges, in any order (cnt ends at zero).
__global__ __launch_bounds__(kBlock) void k_inc_place(int64_t n, const int32_t *__restrict__ connE,
                                                     const int32_t *__restrict__ inc_ptr, int32_t *__restrict__ cnt,
                                                     int32_t *__restrict__ any) {
    const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (q >= n) return;
    const int a = connE[q];
    any[inc_ptr[a] + atomicSub(&cnt[a], 1) - 1] = (int32_t)q;
}

// Each incidence to its rank among its node's (at most a few dozen, in L2).
template <int NPE>
__global__ __launch_bounds__(kBlock) void k_inc_rank(int n_el, const int32_t *__restrict__ connE,
                                                    const int32_t *__restrict__ inc_ptr, const int32_t *__restrict__ any,
                                                    int32_t *__restrict__ inc, int32_t *__restrict__ inc_slot) {
    const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (q >= (int64_t)n_el * NPE) return;
    const int a = connE[q], k0 = inc_ptr[a], k1 = inc_ptr[a + 1];
    int r = k0;
    for (int k = k0; k < k1; ++k) r += any[k] < (int32_t)q;
    inc[r] = (int32_t)q;
    inc_slot[(q % NPE) * n_el + q / NPE] = r;
}

// ----------------------------------------------------------------- pattern ---
// One wave per node a.  Row a's contributions are the pairs (incidence of a,
// local node j): m = valence x NPE of them, at cbase = inc_ptr[a] NPE.  Each
// goes to its place in the order of (column, incidence, j), found by counting
// the entries before it: m^2 comparisons, 60^2 for an average mid node of a
// Tet10 box and 240^2 for its vertices, NV entries per lane against broadcast
// reads of four columns from LDS (one entry and one column at a time: 255 us at
// 20,295 nodes instead of 66).  Rows of more than kRowCap entries (nodes of more
// than 102 Tet10, 256 Tet4 or 128 Hex8 elements) are listed for k_row_sort_large.
constexpr int kRowCap = 1024, kRowWaves = 4;
// flags: an element's J is not constant; nodes of no element; large rows, their entries
enum { kNotAffine, kOrphans, kLargeRows, kLargeEntries, kFlags = 8 };

// where the entries t0 + lane + 64 j of the m in cols[] belong
template <int NV> __device__ __forceinline__ void row_places(const int32_t *cols, int m, int t0, int (&at)[NV], int (&first)[NV]) {
    int32_t v[NV];
    int same[NV];
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int t = t0 + lane + 64 * j;
        v[j] = t < m ? cols[t] : INT32_MAX;
        at[j] = same[j] = 0;
    }
#pragma unroll 2
    for (int u = 0; u < m; u += 4) {  // padded to a multiple of four with INT32_MAX
        const int4 x = *(const int4 *)(cols + u);
        const int32_t xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                at[j] += xs[i] < v[j];
                same[j] += xs[i] == v[j] && u + i < t0 + lane + 64 * j;
            }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        at[j] += same[j];
        first[j] = same[j] == 0;
    }
}

template <int NPE>
__global__ __launch_bounds__(64 * kRowWaves) void k_row_sort(int N, const int32_t *__restrict__ inc_ptr,
                                                            const int32_t *__restrict__ inc,
                                                            const int32_t *__restrict__ connE, int32_t *__restrict__ sorted,
                                                            int32_t *__restrict__ contrib, int32_t *__restrict__ rowlen,
                                                            int32_t *__restrict__ flags, int2 *__restrict__ large) {
    __shared__ __attribute__((aligned(16))) int32_t rows[kRowWaves][kRowCap];
    const int lane = threadIdx.x & 63;
    const int a = blockIdx.x * kRowWaves + (threadIdx.x >> 6);
    int32_t *cols = rows[threadIdx.x >> 6];
    const int k0 = a < N ? inc_ptr[a] : 0, m = a < N ? (inc_ptr[a + 1] - k0) * NPE : 0;
    const bool lds = m <= kRowCap;
    if (lds)
        for (int t = lane; t < ((m + 3) & ~3); t += 64)
            cols[t] = t < m ? connE[(int64_t)(inc[k0 + t / NPE] / NPE) * NPE + t % NPE] : INT32_MAX;
    __syncthreads();
    int distinct = 0;
    const int64_t base = (int64_t)k0 * NPE;
    auto put = [&](int t, int at, int first, int32_t v) {
        sorted[base + at] = v;
        contrib[base + at] = inc[k0 + t / NPE] * NPE + t % NPE;
        distinct += first;
    };
    if (!lds) {
        if (lane == 0) large[atomicAdd(flags + kLargeRows, 1)] = {a, atomicAdd(flags + kLargeEntries, m)};
    } else if (m <= 64) {
        int at[1], first[1];
        row_places<1>(cols, m, 0, at, first);
        if (lane < m) put(lane, at[0], first[0], cols[lane]);
    } else {
        for (int t0 = 0; t0 < m; t0 += 256) {
            int at[4], first[4];
            row_places<4>(cols, m, t0, at, first);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = t0 + lane + 64 * j;
                if (t < m) put(t, at[j], first[j], cols[t]);
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) distinct += __shfl_xor(distinct, off, 64);
    if (lane == 0 && a < N) {
        rowlen[a] = distinct;
        if (m == 0) atomicAdd(flags + kOrphans, 1);
    }
}

// One workgroup per listed row: its entries as keys (column, t), sorted in LDS in
// runs of kRun and merged in memory, run by run with its neighbour, each key to its
// own place plus the smaller keys of the other run (a binary search).  At 1,922
// Tet4 around a node (7,688 entries) the upload takes 0.7 ms instead of 142 with
// the comparison of all pairs in one wave, at 968 Tet10 0.64 instead of 299.
// `keys`: two arrays of `entries`.
constexpr int kRun = 4096, kLargeThreads = 1024;
template <int NPE>
__global__ __launch_bounds__(kLargeThreads) void k_row_sort_large(const int2 *__restrict__ large, int64_t entries,
                                                                 const int32_t *__restrict__ inc_ptr,
                                                                 const int32_t *__restrict__ inc,
                                                                 const int32_t *__restrict__ connE, uint64_t *keys,
                                                                 int32_t *__restrict__ sorted, int32_t *__restrict__ contrib,
                                                                 int32_t *__restrict__ rowlen) {
    __shared__ uint64_t run[kRun];
    const int a = large[blockIdx.x].x, k0 = inc_ptr[a], m = (inc_ptr[a + 1] - k0) * NPE;
    uint64_t *from = keys + large[blockIdx.x].y, *to = from + entries;
    for (int r0 = 0; r0 < m; r0 += kRun) {
        const int n = min(kRun, m - r0);
        int n2 = 2;
        while (n2 < n) n2 <<= 1;
        for (int i = threadIdx.x; i < n2; i += kLargeThreads) {
            const int t = r0 + i;
            run[i] = i < n ? (uint64_t)(uint32_t)connE[(int64_t)(inc[k0 + t / NPE] / NPE) * NPE + t % NPE] << 32 | (uint32_t)t : ~0ull;
        }
        sort_keys<kLargeThreads>(run, n2);
        for (int i = threadIdx.x; i < n; i += kLargeThreads) from[r0 + i] = run[i];
        __syncthreads();
    }
    for (int64_t w = kRun; w < m; w *= 2) {
        for (int i = threadIdx.x; i < m; i += kLargeThreads) {
            const uint64_t v = from[i];
            const int64_t r = i / w, o0 = min((r ^ 1) * w, (int64_t)m), o1 = min(((r ^ 1) + 1) * w, (int64_t)m);
            int64_t lo = o0, hi = o1;  // the first key of the other run above v
            while (lo < hi) {
                const int64_t mid = (lo + hi) / 2;
                if (from[mid] < v) lo = mid + 1;
                else hi = mid;
            }
            to[(r & ~(int64_t)1) * w + (i - r * w) + (lo - o0)] = v;
        }
        __syncthreads();
        uint64_t *const swap = from;
        from = to;
        to = swap;
    }
    const int64_t base = (int64_t)k0 * NPE;
    int distinct = 0, total;
    for (int i = threadIdx.x; i < m; i += kLargeThreads) {
        const uint64_t v = from[i];
        const int t = (int)(uint32_t)v;
        sorted[base + i] = (int32_t)(v >> 32);
        contrib[base + i] = inc[k0 + t / NPE] * NPE + t % NPE;
        distinct += i == 0 || from[i - 1] >> 32 != v >> 32;
    }
    (void)block_scan<kLargeThreads>(distinct, &total);
    if (threadIdx.x == 0) rowlen[a] = total;
}

// One wave per node: the row's columns and the blocks' ranges of contributions
// from the sorted columns.
__global__ __launch_bounds__(kBlock) void k_row_write(int N, int npe, const int32_t *__restrict__ inc_ptr,
                                                     const int32_t *__restrict__ sorted, const int32_t *__restrict__ brow,
                                                     int32_t *__restrict__ bcol, int32_t *__restrict__ blk_row,
                                                     int32_t *__restrict__ cptr, int32_t *__restrict__ bdiag) {
    const int lane = threadIdx.x & 63, a = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    if (a >= N) return;
    const int64_t base = (int64_t)inc_ptr[a] * npe;
    const int m = (inc_ptr[a + 1] - inc_ptr[a]) * npe;
    int s0 = brow[a];
    if (m == 0 && lane == 0) bdiag[a] = s0;
    for (int t0 = 0; t0 < m; t0 += 64) {
        const int t = t0 + lane;
        const int32_t v = t < m ? sorted[base + t] : -1;
        const bool head = t < m && (t == 0 || sorted[base + t - 1] != v);
        const unsigned long long hm = __ballot(head);
        if (head) {
            const int s = s0 + __popcll(hm & ((1ull << lane) - 1));
            bcol[s] = v;
            blk_row[s] = a;
            cptr[s] = (int32_t)(base + t);
            if (v == a) bdiag[a] = s;
        }
        s0 += __popcll(hm);
    }
    if (a == N - 1 && lane == 0) cptr[brow[N]] = (int32_t)(base + m);
}

// Tet10 edge mid nodes at their edge midpoints (and Hex8 parallelepipeds) make
// J constant over the element; one factor set per element then suffices.
template <int NPE>
__global__ __launch_bounds__(kBlock) void k_not_affine(int n_el, const int32_t *__restrict__ conn, const double *__restrict__ X,
                                                      int32_t *__restrict__ flags) {
    const int e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= n_el) return;
    double P[NPE][3];
#pragma unroll
    for (int i = 0; i < NPE; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) P[i][k] = X[3 * (size_t)conn[(size_t)i * n_el + e] + k];
    double h = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) h = fmax(h, fabs(P[1][k] - P[0][k]));
    const double tol = 1e-12 * fmax(h, 1e-300);
    bool bad = false;
    if constexpr (NPE == 10) {
        constexpr int ed[6][2] = {{0, 1}, {1, 2}, {2, 0}, {0, 3}, {1, 3}, {2, 3}};
#pragma unroll
        for (int m = 0; m < 6; ++m)
#pragma unroll
            for (int k = 0; k < 3; ++k) bad = bad || fabs(P[4 + m][k] - 0.5 * (P[ed[m][0]][k] + P[ed[m][1]][k])) > tol;
    } else {  // Hex8: x_i = x0 + sum of the three edge vectors it spans
        constexpr int s[8][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0}, {0, 0, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 1}};
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                double v = P[0][k];
                if (s[i][0]) v += P[1][k] - P[0][k];
                if (s[i][1]) v += P[3][k] - P[0][k];
                if (s[i][2]) v += P[4][k] - P[0][k];
                bad = bad || fabs(P[i][k] - v) > tol * 8;
            }
    }
    if (bad) flags[kNotAffine] = 1;
}

// ----------------------------------------------------------------- launches ---
// the arrays in the scratch of an upload
namespace {
struct ListScratch {
    int32_t *connE, *any, *cnt, *flags, *rowlen, *bsum, *sorted;  // by element, placed incidences, counts, flags, ...
    int2 *large;                                                  // large rows: node, first key
    int64_t total;
    ListScratch(int32_t *p, int64_t N, int64_t n_el, int npe) {
        const int64_t q = n_el * npe;
        int64_t at = 0;
        auto take = [&](int64_t n) {
            int32_t *r = p ? p + at : nullptr;
            at += n;
            return r;
        };
        large = (int2 *)take(2 * (q * npe / kRowCap + 1));  // first: its alignment
        connE = take(q);
        any = take(q);
        cnt = take(N);
        flags = take(kFlags);
        rowlen = take(N);
        bsum = take((N + kScan - 1) / kScan);
        sorted = take(q * npe);
        total = at;
    }
    ListScratch(jfm_ctx *ctx, int32_t *p) : ListScratch(p, ctx->N, ctx->n_el, ctx->npe) {}
};
}  // namespace

int64_t mesh_lists_scratch(int64_t N, int64_t n_el, int npe) { return ListScratch(nullptr, N, n_el, npe).total; }

template <int NPE> static void incidences(jfm_ctx *ctx, const ListScratch &L) {
    hipStream_t s = ctx->stream;
    const int N = (int)ctx->N, n_el = (int)ctx->n_el;
    const int64_t q = (int64_t)n_el * NPE;
    const unsigned gq = (unsigned)((q + kBlock - 1) / kBlock);
    if (gq) k_conn_split<NPE><<<gq, kBlock, 0, s>>>(n_el, L.connE, ctx->conn, L.cnt);
    scan(s, N, L.cnt, ctx->inc_ptr, L.bsum);
    if (gq) {
        k_inc_place<<<gq, kBlock, 0, s>>>(q, L.connE, ctx->inc_ptr, L.cnt, L.any);
        k_inc_rank<NPE><<<gq, kBlock, 0, s>>>(n_el, L.connE, ctx->inc_ptr, L.any, ctx->inc, ctx->inc_slot);
    }
    k_row_sort<NPE><<<(N + kRowWaves - 1) / kRowWaves, 64 * kRowWaves, 0, s>>>(N, ctx->inc_ptr, ctx->inc, L.connE, L.sorted,
                                                                             ctx->contrib, L.rowlen, L.flags, L.large);
    scan(s, N, L.rowlen, ctx->brow, L.bsum);
    if constexpr (NPE != 4)
        if (gq) k_not_affine<NPE><<<(n_el + kBlock - 1) / kBlock, kBlock, 0, s>>>(n_el, ctx->conn, ctx->X, L.flags);
}

hipError_t launch_mesh_lists(jfm_ctx *ctx, int32_t *scratch, MeshFlags *flags) {
    const int64_t q = ctx->n_el * ctx->npe;
    hipStream_t s = ctx->stream;
    const ListScratch L(ctx, scratch);
    hipError_t e = hipMemsetAsync(L.cnt, 0, 4 * (size_t)(ctx->N + kFlags), s);  // and the flags
    if (e == hipSuccess && q) e = hipMemcpyAsync(L.connE, ctx->h_conn.data(), 4 * (size_t)q, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    switch (ctx->npe) {
    case 10: incidences<10>(ctx, L); break;
    case 4: incidences<4>(ctx, L); break;
    case 8: incidences<8>(ctx, L); break;
    default: return hipErrorInvalidValue;
    }
    int32_t got[4] = {0, 0, 0, 0};
    if ((e = hipGetLastError()) == hipSuccess) e = hipMemcpyAsync(got, L.flags, sizeof got, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(&flags->nnzb, ctx->brow + ctx->N, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    flags->affine = got[kNotAffine] == 0;
    flags->orphans = got[kOrphans];
    flags->large_rows = got[kLargeRows];
    flags->large_entries = got[kLargeEntries];
    return e;
}

hipError_t launch_large_rows(jfm_ctx *ctx, int32_t *scratch, uint64_t *keys, MeshFlags *flags) {
    hipStream_t s = ctx->stream;
    const ListScratch L(ctx, scratch);
    auto sort = [&](auto kernel) {
        kernel<<<(unsigned)flags->large_rows, kLargeThreads, 0, s>>>(L.large, flags->large_entries, ctx->inc_ptr, ctx->inc, L.connE, keys,
                                                                     L.sorted, ctx->contrib, L.rowlen);
    };
    switch (ctx->npe) {
    case 10: sort(k_row_sort_large<10>); break;
    case 4: sort(k_row_sort_large<4>); break;
    case 8: sort(k_row_sort_large<8>); break;
    default: return hipErrorInvalidValue;
    }
    scan(s, (int)ctx->N, L.rowlen, ctx->brow, L.bsum);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&flags->nnzb, ctx->brow + ctx->N, 4, hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);  // also before the keys go
    return e == hipSuccess ? w : e;
}

hipError_t launch_pattern_write(jfm_ctx *ctx, int32_t *scratch) {
    const ListScratch L(ctx, scratch);
    k_row_write<<<(unsigned)((ctx->N + 3) / 4), kBlock, 0, ctx->stream>>>((int)ctx->N, ctx->npe, ctx->inc_ptr, L.sorted, ctx->brow, ctx->bcol,
                                                                          ctx->blk_row, ctx->cptr, ctx->bdiag);
    return hipGetLastError();
}

}  // namespace jfem
