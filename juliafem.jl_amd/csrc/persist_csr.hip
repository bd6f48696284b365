// persist_csr.hip -- the resident PCG on the assembled matrix (gfx950).
//
// As persist.hip, one kernel is the whole solve; here a workgroup keeps a run of
// consecutive nodes (their rows of K).  Launched, an iteration took 12.4 us at
// 6,048 DOFs (Hex8) and 21.3 at 61,347 (Tet10): product, update and direction,
// each bound by its launch and its dependent loads; resident they take 6.7 and
// 13.1 us, most of it the two exchanges' latency.  A workgroup's vectors at its own nodes are in registers;
// of p it keeps a copy in LDS at every node that its rows have columns for:
//
//   z = M r; z of the own nodes out; partials of (r.z, r.r)  -> exchange C
//   p = z + beta p at the own nodes and at the others' (z read)
//   q = K p: lanes of a wave share a node's blocks; p.q     -> exchange B
//   x += alpha p, r -= alpha q
//
// The copies of p at a node are updated with the same operations from the same
// values, so they stay equal to the bit.  z is stored (and waited for) before
// the scalars of exchange C that its readers wait for, and written again only
// after exchange B, which a workgroup enters when it has read it.  A lane keeps
// its first two blocks of the matrix in registers (19 MB over the chip, FP64); the
// others are read from the caches each iteration, always by the same workgroup,
// so they stay in its XCD's L2.
#include <algorithm>

#include "persist_exchange.h"
#include "sort_scan.h"

namespace jfem {

constexpr int kRT = 512;                 // threads
// Own nodes of a workgroup: 32 while the workgroups suffice (16, 32 and 64: 6.97,
// 6.74 and 7.41 us per iteration at 2,016 nodes, 7.16, 6.51 and 6.37 at 2,989), and
// at most 128, four lanes per row.  Beyond that the launched product, with four
// times the waves per CU, hides the matrix' latency better: FP64 17.3 against 24.1
// us at 27,225 nodes, 27.8 against 27.1 at 32,895 (two lanes per row).
constexpr int kRowNodes = 32, kRowsMaxNodes = 128 * kPersistPatches;
constexpr int kLocal = 3072;             // most nodes with columns in a workgroup's rows (FP64: 72 KB)
constexpr int kHalo = kLocal / kRT;
constexpr int kKeep = 2;                 // blocks of a lane in registers (none: 8.2 us at 2,016 nodes)

// One workgroup's columns as a set of bits: their nodes in ascending order to
// loc[], and each block's position among them to lcol[].
__global__ __launch_bounds__(kRT) void k_rows_setup(int N, int per, const int32_t *__restrict__ brow,
                                                   const int32_t *__restrict__ bcol, int32_t *__restrict__ nloc,
                                                   int32_t *__restrict__ loc, uint16_t *__restrict__ lcol,
                                                   int32_t *__restrict__ bad) {
    constexpr int kWords = kRowsMaxNodes / 32, kPer = kWords / kRT;
    __shared__ uint32_t bits[kWords];
    __shared__ int before[kWords];
    const int g = blockIdx.x, t = threadIdx.x, n0 = min(g * per, N), n1 = min(n0 + per, N);
    for (int w = t; w < kWords; w += kRT) bits[w] = 0;
    __syncthreads();
    for (int a = n0 + t; a < n1; a += kRT) atomicOr(&bits[a >> 5], 1u << (a & 31));
    const int s0 = brow[n0], s1 = brow[n1];
    for (int s = s0 + t; s < s1; s += kRT) atomicOr(&bits[bcol[s] >> 5], 1u << (bcol[s] & 31));
    __syncthreads();
    int mine = 0, total;
    for (int j = 0; j < kPer; ++j) mine += __popc(bits[t * kPer + j]);
    int at = block_scan<kRT>(mine, &total);
    for (int j = 0; j < kPer; ++j) {
        const int w = t * kPer + j;
        before[w] = at;
        at += __popc(bits[w]);
    }
    __syncthreads();
    if (total > kLocal) {  // uniform
        if (t == 0) {
            nloc[g] = 0;
            *bad = 1;
        }
        return;
    }
    if (t == 0) nloc[g] = total;
    for (int w = t; w < kWords; w += kRT) {
        int k = before[w];
        for (uint32_t b = bits[w]; b; b &= b - 1) loc[(size_t)g * kLocal + k++] = 32 * w + __ffs(b) - 1;
    }
    for (int s = s0 + t; s < s1; s += kRT) {
        const int c = bcol[s];
        lcol[s] = (uint16_t)(before[c >> 5] + __popc(bits[c >> 5] & ((1u << (c & 31)) - 1)));
    }
}

template <typename T> struct RowsArgs {
    int N, nwg, per;
    const int32_t *brow, *nloc, *loc;
    const uint16_t *lcol;
    const T *vals;
    const uint8_t *fixed;
    const T *Minv, *b, *x0, *r0;  // the start and its true residual (null: from 0)
    T *x;                     // (not x0)
    void *z;                  // 4 values per node
    uint64_t *words;
    double rtol2;
    int maxit, polls;
    PcgScalars *S;
};

template <typename T>
__global__ __launch_bounds__(kRT, 2) void k_pcg_rows(const RowsArgs<T> A0) {
    __shared__ T ps[3 * kLocal];
    __shared__ T qs[3 * kRT];
    __shared__ GridSumLds<1> shB;
    __shared__ GridSumLds<2> shC;
    __shared__ int bad;
    const RowsArgs<T> &A = A0;
    const int g = (int)blockIdx.x, t = (int)threadIdx.x, nwg = A.nwg;
    const int n0 = min(g * A.per, A.N), nown = min(n0 + A.per, A.N) - n0, nloc = A.nloc[g];
    const int32_t *loc = A.loc + (size_t)g * kLocal;
    uint64_t *wordsB = A.words, *wordsC = wordsB + grid_words(1, nwg, true);
    const Partials<T> zb(A.z, A.N);
    if (t == 0) bad = 0;
    const bool own = t < nown;
    const int node = own ? n0 + t : 0;
    // the nodes this thread reads z of (not the own ones), and where the own ones are
    int halo[kHalo];
    __shared__ int own0;
#pragma unroll
    for (int j = 0; j < kHalo; ++j) {
        const int l = t + j * kRT, a = l < nloc ? loc[l] : -1;
        if (a == n0) own0 = l;
        halo[j] = a >= n0 && a < n0 + nown ? -1 : a;
    }
    for (int l = t; l < 3 * nloc; l += kRT) ps[l] = T(0);
    // a row's blocks over LN lanes, every row at once
    int LN = kRT / (kRowsMaxNodes / kPersistPatches);
    while (LN < 32 && 2 * LN * nown <= kRT) LN *= 2;
    const int lane = t & (LN - 1), row = t / LN;
    const bool has_row = row < nown;
    const int s0 = has_row ? A.brow[n0 + row] : 0,
              nb = has_row ? A.brow[n0 + row + 1] - s0 : 0, rs = 3 * nb;
    const T *vals = A.vals + 9 * (size_t)s0;
    T kv[kKeep][9];   // its first blocks stay in registers
    int kc[kKeep];
#pragma unroll
    for (int j = 0; j < kKeep; ++j) {
        const int k = lane + LN * j;
        kc[j] = k < nb ? 3 * (int)A.lcol[s0 + k] : 0;
#pragma unroll
        for (int c = 0; c < 9; ++c) kv[j][c] = k < nb ? vals[c / 3 * rs + 3 * k + c % 3] : T(0);
    }
    T M[9], r[3], x[3];
    uint32_t fx = 0;
#pragma unroll
    for (int m = 0; m < 9; ++m) M[m] = own ? A.Minv[9 * (size_t)node + m] : T(0);
    double bb[1] = {0.0};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t d = 3 * (size_t)node + c;
        if (own && A.fixed && A.fixed[d]) fx |= 1u << c;
        const T bv = own ? A.b[d] : T(0);
        bb[0] += (double)bv * (double)bv;
        r[c] = own && A.r0 ? A.r0[d] : bv;
        x[c] = own && A.r0 ? A.x0[d] : T(0);
    }
    __syncthreads();  // bad, own0, ps
    const int me = 3 * (own0 + t);
    uint32_t epoch = 1;
    if (!grid_sum<1, kRT, true>(bb, wordsB, g, nwg, epoch, A.polls, shB, &bad)) {
        if (t == 0) A.S->fail = 1;
        return;
    }
    const double tol2 = A.rtol2 * bb[0];
    double rz = 0.0, rr = 0.0, rr0 = 0.0, pq = 1.0, alpha_d = 0.0, beta_d = 0.0;
    int it = 0, done = DONE_RUNNING;
    for (;;) {
        T z[3];
        double s2[2] = {0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            z[c] = M[3 * c] * r[0] + M[3 * c + 1] * r[1] + M[3 * c + 2] * r[2];
            s2[0] += (double)r[c] * (double)z[c];
            s2[1] += (double)r[c] * (double)r[c];
        }
        ++epoch;
        if (own) zb.template put<3>(node, z);
        stores_done();  // before the block barrier in grid_sum, hence before its words
        if (!grid_sum<2, kRT, true>(s2, wordsC, g, nwg, epoch, A.polls, shC, &bad)) break;
        rr = s2[1];
        if (epoch == 2) rr0 = rr;  // the start
        else ++it;
        if (rr <= tol2) {  // the same in every workgroup
            done = DONE_CONVERGED;
            break;
        }
        if (epoch > 2) {
            beta_d = s2[0] / rz;
            if (!(pq > 0.0) || !(s2[0] > 0.0) || !finite(s2[0])) done = DONE_BREAKDOWN;
            else if (it >= A.maxit) done = DONE_MAXIT;
        }
        rz = s2[0];
        if (done) break;
        // p = z + beta p at every node of the rows' columns
        const T beta = (T)beta_d;
        T zh[kHalo][3];
#pragma unroll
        for (int j = 0; j < kHalo; ++j)
            if (halo[j] >= 0) zb.template get<3>(halo[j], zh[j]);
#pragma unroll
        for (int j = 0; j < kHalo; ++j)
            if (halo[j] >= 0) {
                T *p = ps + 3 * (t + j * kRT);
#pragma unroll
                for (int c = 0; c < 3; ++c) p[c] = zh[j][c] + beta * p[c];
            }
        T pv[3] = {T(0), T(0), T(0)};
        if (own)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                pv[c] = z[c] + beta * ps[me + c];
                ps[me + c] = pv[c];
            }
        __syncthreads();
        T a0 = T(0), a1 = T(0), a2 = T(0);
        auto add = [&](const T (&v)[9], int l) {
            const T p0 = ps[l], p1 = ps[l + 1], p2 = ps[l + 2];
            a0 += v[0] * p0 + v[1] * p1 + v[2] * p2;
            a1 += v[3] * p0 + v[4] * p1 + v[5] * p2;
            a2 += v[6] * p0 + v[7] * p1 + v[8] * p2;
        };
#pragma unroll
        for (int j = 0; j < kKeep; ++j) add(kv[j], kc[j]);
#pragma unroll 2
        for (int k = lane + LN * kKeep; k < nb; k += LN) {
            T v[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) v[c] = vals[c / 3 * rs + 3 * k + c % 3];
            add(v, 3 * (int)A.lcol[s0 + k]);
        }
        for (int off = LN / 2; off > 0; off >>= 1) {
            a0 += __shfl_xor(a0, off, 64);
            a1 += __shfl_xor(a1, off, 64);
            a2 += __shfl_xor(a2, off, 64);
        }
        if (has_row && lane == 0) {
            qs[3 * row] = a0;
            qs[3 * row + 1] = a1;
            qs[3 * row + 2] = a2;
        }
        __syncthreads();
        T q[3];
        double e1[1] = {0.0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            q[c] = own && !(fx >> c & 1u) ? qs[3 * t + c] : T(0);
            e1[0] += (double)pv[c] * (double)q[c];
        }
        if (!grid_sum<1, kRT, true>(e1, wordsB, g, nwg, epoch, A.polls, shB, &bad)) break;
        pq = e1[0];
        alpha_d = (pq > 0.0 && finite(pq)) ? rz / pq : 0.0;
        const T alpha = (T)alpha_d;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            x[c] += alpha * pv[c];
            r[c] -= alpha * q[c];
        }
    }
    if (bad) {
        if (t == 0) A.S->fail = 1;
        return;
    }
    if (own)
#pragma unroll
        for (int c = 0; c < 3; ++c) A.x[3 * (size_t)node + c] = x[c];
    if (g == 0 && t == 0) {
        PcgScalars *S = A.S;
        S->rz[0] = S->rz[1] = rz;
        S->alpha = alpha_d;
        S->beta = beta_d;
        S->pq = pq;
        S->rr = rr;
        S->rr0 = rr0;
        S->bb = bb[0];
        S->tol2 = tol2;
        S->iter = it;
        S->done[0] = S->done[1] = done;
    }
}

// ------------------------------------------------------------------- host ---
bool jfem_rows_maybe(const jfm_ctx *ctx) {
    return ctx->N <= kRowsMaxNodes && ctx->cus >= kPersistPatches && ctx->n_el > 0 &&
           (!ctx->rows.ready || ctx->rows.usable);
}

// Once per mesh; rows.usable tells whether every workgroup's columns fit.
int jfem_rows_setup(jfm_ctx *ctx) {
    auto &R = ctx->rows;
    if (R.ready) return JFM_OK;
    R.ready = true;
    R.usable = false;
    const int N = (int)ctx->N;
    R.per = std::max(kRowNodes, (N + kPersistPatches - 1) / kPersistPatches);
    R.nwg = (N + R.per - 1) / R.per;
    hipStream_t s = ctx->stream;
    int32_t *d_bad = jfm_alloc<int32_t>(ctx, 1), got = 0;
    const bool ok = d_bad && (R.nloc = jfm_alloc<int32_t>(ctx, R.nwg)) &&
                    (R.loc = jfm_alloc<int32_t>(ctx, (int64_t)R.nwg * kLocal)) &&
                    (R.lcol = jfm_alloc<uint16_t>(ctx, ctx->nnzb)) && (R.z = jfm_alloc<double>(ctx, 4 * (int64_t)N)) &&
                    (R.words = jfm_alloc<uint64_t>(ctx, grid_words(1, R.nwg, true) + grid_words(2, R.nwg, true)));
    if (!ok) {
        jfm_free(ctx, d_bad);
        jfem_rows_release(ctx);
        return jfm_fail(ctx, JFM_ENOMEM, "resident PCG allocation failed");
    }
    hipError_t e = hipMemsetAsync(d_bad, 0, 4, s);
    if (e == hipSuccess) {
        k_rows_setup<<<R.nwg, kRT, 0, s>>>(N, R.per, ctx->brow, ctx->bcol, R.nloc, R.loc, R.lcol, d_bad);
        e = hipMemcpyAsync(&got, d_bad, 4, hipMemcpyDeviceToHost, s);
    }
    const hipError_t w = hipStreamSynchronize(s);
    jfm_free(ctx, d_bad);
    if (e == hipSuccess) e = w;
    if (e != hipSuccess || got) {
        jfem_rows_release(ctx);
        R.ready = true;
        return e == hipSuccess ? JFM_OK : jfm_hip_fail(ctx, e, "resident PCG rows");
    }
    R.usable = true;
    return JFM_OK;
}

void jfem_rows_release(jfm_ctx *ctx) {
    auto &R = ctx->rows;
    for (void *p : {(void *)R.nloc, (void *)R.loc, (void *)R.lcol, (void *)R.z, (void *)R.words}) jfm_free(ctx, p);
    R = {};
}

template <typename T>
hipError_t launch_pcg_rows(jfm_ctx *ctx, const T *Minv, const T *b, const T *x0, const T *r0, T *x, double rtol, int maxit) {
    const auto &R = ctx->rows;
    RowsArgs<T> A{};
    A.N = (int)ctx->N;
    A.nwg = R.nwg;
    A.per = R.per;
    A.brow = ctx->brow;
    A.nloc = R.nloc;
    A.loc = R.loc;
    A.lcol = R.lcol;
    if constexpr (sizeof(T) == 8)
        A.vals = ctx->vals64;
    else
        A.vals = ctx->vals32;
    A.fixed = ctx->fixed;
    A.Minv = Minv;
    A.b = b;
    A.x0 = x0;
    A.r0 = r0;
    A.x = x;
    A.z = R.z;
    A.words = R.words;
    A.rtol2 = rtol * rtol;
    A.maxit = maxit;
    A.polls = ctx->persist_polls;
    A.S = ctx->S;
    launch_persist_clear(ctx, grid_words(1, R.nwg, true) + grid_words(2, R.nwg, true), R.words, 0, nullptr, 1, A.S);
    k_pcg_rows<T><<<R.nwg, kRT, 0, ctx->stream>>>(A);
    return hipGetLastError();
}

template hipError_t launch_pcg_rows<double>(jfm_ctx *, const double *, const double *, const double *, const double *, double *, double, int);
template hipError_t launch_pcg_rows<float>(jfm_ctx *, const float *, const float *, const float *, const float *, float *, double, int);

}  // namespace jfem
