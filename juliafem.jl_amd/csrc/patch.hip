// patch.hip -- fused matrix-free K.u over element patches (gfx950).
//
// The two-phase operator (fem_kernels.hip) writes every element's 3 x npe
// terms to HBM and reads them back in the nodal gather.  Here the elements are
// ordered along a Morton curve of their centroids and cut into patches of
// kPatch = 480 (one workgroup each, one element per thread).  A workgroup computes its
// elements' terms with the same element product (mf_element.h) into LDS and
// then sums them per patch node, in ascending local element order, from a
// patch-local incidence list:
//  * a node whose incidences all lie in the patch (interior) is finished and
//    written to y directly;
//  * any other node writes the patch's partial sum to a slot; a second kernel
//    adds each such node's partials in ascending patch order.
// Every node is written exactly once (nodes of no element through the second
// kernel, as zero), there are no floating-point atomics and the result does
// not depend on the launch: the order of every sum is fixed by the patch
// structure.  The result equals the two-phase operator's up to the order of
// the nodal sums.
//
// Reference: the operator of ext/JuliaFEMCUDAExt.jl:179-193 / 293-361 (element
// loop and nodal assembly), elements per src/problems_elasticity.jl:203-451.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "ebe_element.h"
#include "mf_element.h"
#include "sort_scan.h"

namespace jfem {

// Elements per patch = threads per workgroup.  The LDS image (57.6 KB FP32,
// 115 KB FP64 for Tet10) allows two workgroups per CU, so the patch count is
// best a multiple of 2 x 256: 480 gives exactly 512 patches for 245,760
// elements and 4,096 for 1,966,080 (512 elements: 480 patches, 32 CUs with
// one, and 4% slower).
constexpr int kPatch = kPatchElems;

// Fused element product and patch-local nodal sums.  LDS holds the patch's
// element terms as ys[(3 i + c) * kPatch + local element].  The patch's nodes
// are taken in rounds of kPatch, one per thread; round q lists the j-th
// incidence of its thread t's node at linT[rbase[q] + j kPatch + t] (j below
// the node's count), so the lanes of a wave read consecutive entries.  Nodes
// are sorted by count within a patch, so a round's counts are close; the
// first rounds' node data is loaded before the element product.  A
// shared node's partial sum goes to its slot s (pn_out = -(s + 1)):
// bpart[3 s + c].
// Block partials of y.dotv over the interior nodes go to ppart; with ppart
// and no dotv (affine Tet10 matrix-free form), the block partials of the
// element energies x_e.K_e x_e instead, which sum to x.Kx.
// The element product is the matrix-free one (mf_element.h) from the
// patch-ordered geometric factors el, or with EBE the stored-matrix one
// (ebe_element.h) from element matrices el stored in the patch order.
template <int NPE, typename T, bool AFF, bool EBE, bool C16, bool FOLD>
__global__ __launch_bounds__(kPatch) void k_ku_patch(int n_el, int npatch, int npn, const int32_t *__restrict__ connP,
                                                    const uint16_t *__restrict__ connP16, const int32_t *__restrict__ pbase,
                                                    const T *__restrict__ el, const T *__restrict__ x,
                                                    const int32_t *__restrict__ pn_ptr, const uint16_t *__restrict__ pn_cnt,
                                                    const int32_t *__restrict__ pn_out, const int32_t *__restrict__ rstart,
                                                    const int32_t *__restrict__ rbase, const uint16_t *__restrict__ linT,
                                                    const uint8_t *__restrict__ fixed, T *__restrict__ y,
                                                    T *__restrict__ bpart, const T *__restrict__ dotv,
                                                    double *__restrict__ ppart, const int *__restrict__ done,
                                                    T rho, int xs, int bs) {
    // blockIdx.y: product of vector y of a batch, xs values further (no dotv then)
    x += (size_t)blockIdx.y * xs;
    y += (size_t)blockIdx.y * xs;
    bpart += (size_t)blockIdx.y * bs;
    __shared__ T ys[3 * NPE * kPatch];
    const int p = xcd_block();
    if (p >= npatch) return;  // whole workgroup (grid padded to a multiple of 8)
    const int dn = done ? *done : 0;  // tested once the prefetches below are in flight
    const int t = threadIdx.x;
    const int k = p * kPatch + t;
    // the first kPreR rounds' node data and first incidences, loaded before
    // the element product so that their latency overlaps it
    const int lb = pn_ptr[p], le = pn_ptr[p + 1], q0 = rstart[p];
    constexpr int kPre = 4, kPreR = sizeof(T) == 4 ? 3 : 1;  // FP64: registers are short
    constexpr int kExt = 20;  // round 0's incidences kPre .. kPre + kExt - 1, loaded before the barrier
    const int base0 = lb < le ? rbase[q0] : 0;
    int cnt[kPreR], oo[kPreR], mpre[kPreR][kPre];
    // every index below fits 32 bits: byte offsets from the uniform base
    // pointers keep the per-lane address arithmetic 32-bit
    auto fetch = [&](int r, int l, int &c, int &o, int (&mp)[kPre]) {
        c = load_at<uint16_t>(pn_cnt, 2u * (uint32_t)l);
        o = load_at<int32_t>(pn_out, 4u * (uint32_t)l);
        const int base = rbase[q0 + r];
#pragma unroll
        for (int j = 0; j < kPre; ++j)
            mp[j] = j < c ? (int)load_at<uint16_t>(linT, 2u * (uint32_t)(base + j * kPatch + t)) : 0;
    };
#pragma unroll
    for (int r = 0; r < kPreR; ++r) {
        cnt[r] = 0;
        oo[r] = 0;
#pragma unroll
        for (int j = 0; j < kPre; ++j) mpre[r][j] = 0;
        const int l = lb + r * kPatch + t;
        if (l < le) fetch(r, l, cnt[r], oo[r], mpre[r]);
    }
    if (dn) return;  // uniform
    // p.Kp of the PCG step as the sum of the elements' energies (affine Tet10
    // matrix-free form, when partials are asked for without dotv: the caller
    // guarantees x = 0 on fixed DOFs, so x.(masked Kx) = x.Kx)
    constexpr bool kEnergy = !EBE && AFF && NPE == 10;
    double en = 0.0;
    // local node i's id: 16-bit offsets from the patch's lowest id (C16), or
    // the 32-bit ids
    const int pb = C16 ? pbase[p] : 0;  // uniform
    auto node_of = [&](int i) -> uint32_t {
        if constexpr (C16)
            return (uint32_t)pb + load_at<uint16_t>(connP16, 2u * (uint32_t)(i * n_el + k));
        else
            return (uint32_t)load_at<int32_t>(connP, 4u * (uint32_t)(i * n_el + k));
    };
    auto x_of = [&](int i, T (&v)[3]) {
        const Trip<T> w = load_at<Trip<T>>(x, (uint32_t)(3 * sizeof(T)) * node_of(i));
        v[0] = w.a;
        v[1] = w.b;
        v[2] = w.c;
    };
    if (k < n_el) {
        auto to_lds = [&](int i, T f0, T f1, T f2) {
            ys[(3 * i) * kPatch + t] = f0;
            ys[(3 * i + 1) * kPatch + t] = f1;
            ys[(3 * i + 2) * kPatch + t] = f2;
        };
        if constexpr (EBE) {
            T f[NPE][3];
            ebe_element<NPE, T>(n_el, k, connP, el, x, f);
#pragma unroll
            for (int i = 0; i < NPE; ++i) to_lds(i, f[i][0], f[i][1], f[i][2]);
        } else if constexpr (kEnergy) {
            if (ppart && !dotv) {
                // x.Kx of the element from the values in registers (u = x - x_0,
                // y = K_e u: u.y = x.K_e x since K_e annihilates translations),
                // each node's three products in T, the nodes' sums in FP64
                T xs[NPE][3];
#pragma unroll
                for (int i = 0; i < NPE; ++i) x_of(i, xs[i]);
                mf_element_x<NPE, T, AFF, FOLD>(
                    n_el, k, el,
                    [&](int i, T (&v)[3]) {
                        v[0] = xs[i][0];
                        v[1] = xs[i][1];
                        v[2] = xs[i][2];
                    },
                    [&](int i, T f0, T f1, T f2) {
                        to_lds(i, f0, f1, f2);
                        if (i > 0)
                            en += (double)((xs[i][0] - xs[0][0]) * f0 + (xs[i][1] - xs[0][1]) * f1 +
                                           (xs[i][2] - xs[0][2]) * f2);
                    },
                    rho);
            } else {
                mf_element_x<NPE, T, AFF, FOLD>(n_el, k, el, x_of, to_lds, rho);
            }
        } else
            mf_element_x<NPE, T, AFF, FOLD>(n_el, k, el, x_of, to_lds, rho);
    }
    // Round 0 holds the patch's nodes of most incidences (up to 24 in a Tet10
    // box mesh, so one wave would otherwise load 20 of them one after the
    // other after the barrier): the rest of its incidences, and the fixed
    // flags of the prefetched rounds' finished nodes, are loaded here, once
    // the element product has freed its registers, so that their latency
    // overlaps the barrier.
    int mext[kExt];
    Trip<uint8_t> fxp[kPreR];
    {
        const int c = cnt[0];  // 0 past the patch's nodes
#pragma unroll
        for (int j = 0; j < kExt; ++j)
            mext[j] = kPre + j < c ? (int)load_at<uint16_t>(linT, 2u * (uint32_t)(base0 + (kPre + j) * kPatch + t)) : 0;
#pragma unroll
        for (int r = 0; r < kPreR; ++r)
            fxp[r] = (fixed && oo[r] >= 0 && cnt[r] > 0) ? load_at<Trip<uint8_t>>(fixed, 3u * (uint32_t)oo[r])
                                                         : Trip<uint8_t>{0, 0, 0};
    }
    __syncthreads();
    double dv = en;
    // node l of round r: the sum of its incidences, to y or to its slot
    // (fx: its fixed flags, when loaded above)
    auto node = [&](int r, int l, int c, int o, const int (&mp)[kPre], const Trip<uint8_t> *fx) {
        T s0 = T(0), s1 = T(0), s2 = T(0);
#pragma unroll
        for (int j = 0; j < kPre; ++j)
            if (j < c) {
                const int m = mp[j];  // (3 i) * kPatch + local element
                s0 += ys[m];
                s1 += ys[m + kPatch];
                s2 += ys[m + 2 * kPatch];
            }
        int j1 = kPre;
        if (r == 0) {
#pragma unroll
            for (int j = 0; j < kExt; ++j)
                if (kPre + j < c) {
                    const int m = mext[j];
                    s0 += ys[m];
                    s1 += ys[m + kPatch];
                    s2 += ys[m + 2 * kPatch];
                }
            j1 = kPre + kExt;
        }
        if (c > j1) {
            const int base = rbase[q0 + r];
            for (int j = j1; j < c; ++j) {
                const int m = load_at<uint16_t>(linT, 2u * (uint32_t)(base + j * kPatch + t));
                s0 += ys[m];
                s1 += ys[m + kPatch];
                s2 += ys[m + 2 * kPatch];
            }
        }
        if (o >= 0) {
            const uint32_t b = 3u * (uint32_t)o;
            if (fixed) {
                const Trip<uint8_t> f = fx ? *fx : load_at<Trip<uint8_t>>(fixed, b);
                if (f.a) s0 = T(0);
                if (f.b) s1 = T(0);
                if (f.c) s2 = T(0);
            }
            store_at<Trip<T>>(y, (uint32_t)sizeof(T) * b, Trip<T>{s0, s1, s2});
            if (dotv) {
                const Trip<T> d = load_at<Trip<T>>(dotv, (uint32_t)sizeof(T) * b);
                dv += (double)s0 * (double)d.a + (double)s1 * (double)d.b + (double)s2 * (double)d.c;
            }
        } else {
            store_at<Trip<T>>(bpart, (uint32_t)sizeof(T) * 3u * (uint32_t)(-o - 1), Trip<T>{s0, s1, s2});
        }
    };
#pragma unroll
    for (int r = 0; r < kPreR; ++r) {
        const int l = lb + r * kPatch + t;
        if (l < le) node(r, l, cnt[r], oo[r], mpre[r], &fxp[r]);
    }
    for (int r = kPreR; lb + r * kPatch < le; ++r) {  // patches of more than kPreR rounds
        const int l = lb + r * kPatch + t;
        if (l < le) {
            int c, o, mp[kPre];
            fetch(r, l, c, o, mp);
            node(r, l, c, o, mp, nullptr);
        }
    }
    if (ppart) {
        double v[1] = {dv};
        block_sum_all<1>(v);
        if (t == 0) ppart[p] = v[0];
    }
}

// Nodes shared between patches (and nodes of no element): y = sum of the
// patch partials in slots bptr[b]..bptr[b+1] (ascending patch order).  The
// shared nodes are listed in the order of their first patch and each block
// takes a contiguous chunk, with the XCD mapping of the patch kernel, so that
// most partials are read from the L2 that received them.  Block partials of
// y.dotv also take in a fixed slice of the patch kernel's partials.
template <typename T>
__global__ __launch_bounds__(256) void k_ku_combine(int nb, int chunk, const int32_t *__restrict__ bptr,
                                                   const int32_t *__restrict__ bnode, const T *__restrict__ bpart,
                                                   const uint8_t *__restrict__ fixed, T *__restrict__ y,
                                                   const T *__restrict__ dotv, const double *__restrict__ ppart,
                                                   int npatch, double *__restrict__ part, const int *__restrict__ done,
                                                   int xs, int bs) {
    y += (size_t)blockIdx.y * xs;
    bpart += (size_t)blockIdx.y * bs;
    // the first node's slot range, its first kPre partials, its mask and its
    // dotv values are all in flight before the convergence flag is tested
    // (the grid gives most threads exactly one node)
    constexpr int kPre = 4;
    const int b0 = xcd_block() * chunk, b1 = min(b0 + chunk, nb);
    auto sum_node = [&](int ra, int rb, const Trip<T> (&v)[kPre], int a, const Trip<uint8_t> &f, const Trip<T> &d,
                        double &dv) {
        T s0 = T(0), s1 = T(0), s2 = T(0);
#pragma unroll
        for (int u = 0; u < kPre; ++u)
            if (ra + u < rb) {
                s0 += v[u].a;
                s1 += v[u].b;
                s2 += v[u].c;
            }
        for (int r = ra + kPre; r < rb; ++r) {
            const Trip<T> w = ld3(bpart, r);
            s0 += w.a;
            s1 += w.b;
            s2 += w.c;
        }
        if (f.a) s0 = T(0);
        if (f.b) s1 = T(0);
        if (f.c) s2 = T(0);
        st3(y, a, s0, s1, s2);
        if (dotv) dv += (double)s0 * (double)d.a + (double)s1 * (double)d.b + (double)s2 * (double)d.c;
    };
    auto load_node = [&](int b, int &ra, int &rb, Trip<T> (&v)[kPre], int &a, Trip<uint8_t> &f, Trip<T> &d) {
        ra = bptr[b];
        rb = bptr[b + 1];
        a = bnode[b];
#pragma unroll
        for (int u = 0; u < kPre; ++u) v[u] = ra + u < rb ? ld3(bpart, ra + u) : Trip<T>{T(0), T(0), T(0)};
        f = fixed ? ld3(fixed, a) : Trip<uint8_t>{0, 0, 0};
        d = dotv ? ld3(dotv, a) : Trip<T>{T(0), T(0), T(0)};
    };
    int ra = 0, rb = 0, a = 0;
    Trip<T> v[kPre], d{T(0), T(0), T(0)};
    Trip<uint8_t> f{0, 0, 0};
    const int bf = b0 + (int)threadIdx.x;
    if (bf < b1) load_node(bf, ra, rb, v, a, f, d);
    if (done && *done) return;
    double dv = 0.0;
    if (ppart)
        for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < npatch; q += gridDim.x * blockDim.x) dv += ppart[q];
    if (bf < b1) sum_node(ra, rb, v, a, f, d, dv);
    for (int b = bf + blockDim.x; b < b1; b += blockDim.x) {  // chunks longer than the block
        load_node(b, ra, rb, v, a, f, d);
        sum_node(ra, rb, v, a, f, d, dv);
    }
    if (part) {
        double v[1] = {dv};
        write_partials<1>(v, part);
    }
}

// geometric factors in patch order: dst[(r * n_el) + k] = src[r * n_el + perm[k]]
template <typename T>
__global__ __launch_bounds__(256) void k_permute_gf(int64_t rows, int n_el, const int32_t *__restrict__ perm,
                                                   const T *__restrict__ src, T *__restrict__ dst) {
    const int64_t total = rows * n_el;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = idx / n_el, k = idx - r * n_el;
        dst[idx] = src[r * n_el + perm[k]];
    }
}

// sqrt(cm) invJ in FP32 from the FP64 factors (affine: one set per element),
// cm = 0.2 mu w detJ as the affine Tet10 product scales it
__global__ __launch_bounds__(256) void k_fold_gf(int n_el, const double *__restrict__ gf, float *__restrict__ gq) {
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < 9 * (int64_t)n_el;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = idx / n_el, k = idx - r * n_el;
        gq[idx] = (float)(sqrt(0.2 * gf[10 * (int64_t)n_el + k]) * gf[idx]);
    }
}

hipError_t launch_patch_factors(jfm_ctx *ctx, const int32_t *perm, double *gf64, float *gf32, float *gfQ32) {
    const int64_t rows = (int64_t)ctx->ngf * GF;
    const int n = (int)ctx->n_el;
    k_permute_gf<double><<<1024, 256, 0, ctx->stream>>>(rows, n, perm, ctx->gf64, gf64);
    k_permute_gf<float><<<1024, 256, 0, ctx->stream>>>(rows, n, perm, ctx->gf32, gf32);
    if (gfQ32) k_fold_gf<<<1024, 256, 0, ctx->stream>>>(n, gf64, gfQ32);
    return hipGetLastError();
}

// ------------------------------------------------------------------- setup ---
bool jfem_patch_enabled() {
    static const bool use = [] {
        const char *v = std::getenv("JFEM_PATCH");
        return !(v && v[0] == '0');
    }();
    return use;
}

void jfem_patch_release(jfm_ctx *ctx) {
    for (void **p : {(void **)&ctx->connP, (void **)&ctx->gfP64, (void **)&ctx->gfP32, (void **)&ctx->gfQ32, (void **)&ctx->pn_ptr,
                     (void **)&ctx->pn_cnt, (void **)&ctx->pn_out, (void **)&ctx->rstart, (void **)&ctx->rbase,
                     (void **)&ctx->linT, (void **)&ctx->bptr, (void **)&ctx->bnode,
                     (void **)&ctx->bpart, (void **)&ctx->ppart, (void **)&ctx->eperm, (void **)&ctx->qsrc,
                     (void **)&ctx->connP16, (void **)&ctx->pbase, (void **)&ctx->na_part}) {
        jfm_free(ctx, *p);
        *p = nullptr;
    }
    ctx->patch_ready = ctx->patch_upload = false;
    ctx->npatch = ctx->npn = ctx->nbnode = ctx->nslot = ctx->bmaxcnt = 0;
    ctx->qsrc_gen = -1;
    if (ctx->ke_perm) {  // element matrices stored in the released patch order
        jfm_free(ctx, ctx->Ke);
        jfm_free(ctx, ctx->Ke32);
        ctx->Ke = nullptr;
        ctx->Ke32 = nullptr;
        ctx->ke_perm = nullptr;
    }
}

// The structure is built by one workgroup per patch from the element order
// (morton_order): it sorts the patch's incidences by (node, element, local node)
// in LDS, ranks the nodes by count, and finds the shared ones and their patches
// from their elements' positions.  The patches' lists lie side by side, so the
// kernel runs twice: sizes, their sums, lists.  (On the host this took 7 ms at
// 12,810 Tet10 elements and 118 ms at 245,760; the upload with it takes less
// than without it before.)
constexpr int kPT = 512;                                   // threads
constexpr int kPerThread = (10 * kPatch + kPT - 1) / kPT;  // incidences at most
constexpr int kPKeys = 8192;
static_assert(10 * kPatch <= kPKeys && 3 * 9 * kPatch + kPatch <= 65536, "keys in LDS, 16-bit incidences");

// Per patch its nodes, rounds, incidence entries, slots and shared nodes that it
// holds first; then their exclusive sums.  Rows of npatch + 1.
enum { kNodes, kRounds, kLin, kSlots, kShared, kSizes };

// WRITE = false: the sizes, the patch's lowest node id, in out[0] whether a
// patch's ids span 65,536 or more, in out[1] the most patches of a node, and in
// total the incidence entries of all patches.  WRITE = true: the lists;
// pn_out of a shared node is -(its rank among the node's patches + 1) here.
template <bool WRITE>
__global__ __launch_bounds__(kPT) void k_patch_build(int n_el, int npe, int npatch, const int32_t *__restrict__ conn,
                                                    const int32_t *__restrict__ perm, const int32_t *__restrict__ epos,
                                                    const int32_t *__restrict__ inc_ptr, const int32_t *__restrict__ inc,
                                                    int32_t *__restrict__ sizes, int32_t *__restrict__ pbase,
                                                    int32_t *__restrict__ out, unsigned long long *__restrict__ total_lin,
                                                    uint16_t *__restrict__ pn_cnt, int32_t *__restrict__ pn_out,
                                                    int32_t *__restrict__ pn_node, int32_t *__restrict__ rbase,
                                                    uint16_t *__restrict__ linT, int32_t *__restrict__ first,
                                                    int32_t *__restrict__ bnode, int32_t *__restrict__ bptr) {
    __shared__ uint64_t key[kPKeys];
    __shared__ uint16_t head[10 * kPatch + 1], cnt[10 * kPatch], ranked[10 * kPatch];
    const int p = blockIdx.x, t = threadIdx.x;
    const int k0 = p * kPatch, ne = min(kPatch, n_el - k0), m = ne * npe;
    auto size_of = [&](int what) -> int32_t & { return sizes[(size_t)what * (npatch + 1) + p]; };
    int n2 = 2;
    while (n2 < m) n2 <<= 1;
    for (int idx = t; idx < n2; idx += kPT) {
        uint64_t v = ~0ull;
        if (idx < m) {
            const int i = idx / ne, kl = idx - i * ne;
            v = (uint64_t)(uint32_t)conn[(size_t)i * n_el + perm[k0 + kl]] << 32 | (uint32_t)(kl << 8 | i);
        }
        key[idx] = v;
    }
    sort_keys<kPT>(key, n2);
    // the nodes, ascending: where each one's incidences start
    auto is_head = [&](int idx) { return idx < m && (idx == 0 || key[idx] >> 32 != key[idx - 1] >> 32); };
    int heads = 0, nn;
    for (int j = 0; j < kPerThread; ++j) heads += is_head(kPerThread * t + j);
    int h = block_scan<kPT>(heads, &nn);
    for (int j = 0; j < kPerThread; ++j)
        if (is_head(kPerThread * t + j)) head[h++] = (uint16_t)(kPerThread * t + j);
    if (t == 0) head[nn] = (uint16_t)m;
    __syncthreads();
    for (int q = t; q < nn; q += kPT) cnt[q] = head[q + 1] - head[q];
    __syncthreads();
    // most incidences first, so that a round's counts are close
    for (int q = t; q < nn; q += kPT) {
        const int c = cnt[q];
        int u = 0;
        for (int o = 0; o < nn; ++o) u += cnt[o] > c || (cnt[o] == c && o < q);
        ranked[u] = (uint16_t)q;
    }
    __syncthreads();
    const int rounds = (nn + kPatch - 1) / kPatch;
    int lin = 0;  // the rounds' largest counts
    for (int r = 0; r < rounds; ++r) {
        if (WRITE && t == 0) rbase[size_of(kRounds) + r] = size_of(kLin) + lin * kPatch;
        lin += cnt[ranked[kPatch * r]];
    }
    if (!WRITE && t == 0) {
        const int lo = (int)(key[0] >> 32), hi = (int)(key[m - 1] >> 32);
        size_of(kNodes) = nn;
        size_of(kRounds) = rounds;
        size_of(kLin) = lin * kPatch;
        pbase[p] = lo;
        if (hi - lo >= 65536) out[0] = 1;
        atomicAdd(total_lin, (unsigned long long)lin * kPatch);
    }
    int slots = WRITE ? size_of(kSlots) : 0, shared = WRITE ? size_of(kShared) : 0;
    for (int u0 = 0; u0 < nn; u0 += kPT) {
        const int u = u0 + t, q = u < nn ? ranked[u] : 0;
        const int n = u < nn ? cnt[q] : 0, a = u < nn ? (int)(key[head[q]] >> 32) : 0;
        int total, rank;
        const int b0 = u < nn ? inc_ptr[a] : 0, b1 = u < nn ? inc_ptr[a + 1] : 0;
        patches_of_node<kPT>(n < b1 - b0, b0, b1, npe, kPatch, npatch, p, inc, epos, &total, &rank);
        int sum, num;
        const int so = slots + block_scan<kPT>(rank == 0 ? total : 0, &sum);
        const int bo = shared + block_scan<kPT>(rank == 0, &num);
        slots += sum;
        shared += num;
        if constexpr (WRITE) {
            if (rank == 0) {
                first[a] = so;
                bnode[bo] = a;
                bptr[bo] = so;
            }
            if (u < nn) {
                const int l = size_of(kNodes) + u, r = u / kPatch, at = u - r * kPatch;
                pn_cnt[l] = (uint16_t)n;
                pn_out[l] = rank < 0 ? a : -(rank + 1);
                pn_node[l] = a;
                int base = size_of(kLin);
                for (int o = 0; o < r; ++o) base += cnt[ranked[kPatch * o]] * kPatch;
                for (int j = 0; j < n; ++j) {
                    const uint32_t w = (uint32_t)key[head[q] + j];
                    linT[base + (size_t)j * kPatch + at] = (uint16_t)(3 * (w & 255) * kPatch + (w >> 8));
                }
            }
        } else if (total > 0) {
            atomicMax(out + 1, total);
        }
    }
    if (!WRITE && t == 0) {
        size_of(kSlots) = slots;
        size_of(kShared) = shared;
    }
}

// the exclusive sums of each row of sizes, the total at its end
__global__ __launch_bounds__(1024) void k_patch_sums(int npatch, int32_t *__restrict__ sizes) {
    int32_t *row = sizes + (size_t)blockIdx.x * (npatch + 1);
    int carry = 0;
    for (int b0 = 0; b0 < npatch; b0 += 1024) {
        const int b = b0 + (int)threadIdx.x;
        int total;
        const int ex = block_scan<1024>(b < npatch ? row[b] : 0, &total);
        if (b < npatch) row[b] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) row[npatch] = carry;
}

// pn_out of the shared nodes: -(the slot of the patch's own partial + 1)
__global__ __launch_bounds__(256) void k_patch_slots(int npn, const int32_t *__restrict__ pn_node,
                                                    const int32_t *__restrict__ first, int32_t *__restrict__ pn_out) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l < npn && pn_out[l] < 0) pn_out[l] -= first[pn_node[l]];
}

// the nodes of no element, ascending, after the shared ones; one workgroup
__global__ __launch_bounds__(1024) void k_patch_orphans(int N, const int32_t *__restrict__ inc_ptr, int nslot,
                                                       int32_t *__restrict__ bnode, int32_t *__restrict__ bptr) {
    int carry = 0;
    for (int a0 = 0; a0 < N; a0 += 1024) {
        const int a = a0 + (int)threadIdx.x;
        const bool o = a < N && inc_ptr[a] == inc_ptr[a + 1];
        int total;
        const int at = carry + block_scan<1024>(o, &total);
        if (o) {
            bnode[at] = a;
            bptr[at] = nslot;
        }
        carry += total;
    }
    if (threadIdx.x == 0) bptr[carry] = nslot;
}

// connectivity in the patch order, with 16-bit ids from each patch's lowest
__global__ __launch_bounds__(256) void k_patch_conn(int n_el, int npe, const int32_t *__restrict__ perm,
                                                   const int32_t *__restrict__ conn, const int32_t *__restrict__ pbase,
                                                   int32_t *__restrict__ connP, uint16_t *__restrict__ connP16) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)n_el * npe) return;
    const int i = (int)(q / n_el), k = (int)(q - (int64_t)i * n_el);
    const int a = conn[(size_t)i * n_el + perm[k]];
    connP[q] = a;
    if (connP16) connP16[q] = (uint16_t)(a - pbase[k / kPatch]);
}

// Builds the patch structure for the uploaded mesh (once per mesh).
int jfem_patch_setup(jfm_ctx *ctx) {
    if (ctx->patch_ready) return JFM_OK;
    const int64_t n_el = ctx->n_el, N = ctx->N;
    const int npe = ctx->npe;
    if (n_el == 0) return JFM_OK;
    if ((int64_t)ctx->h_conn.size() != n_el * npe || (int64_t)ctx->h_X.size() != 3 * N)
        return jfm_fail(ctx, JFM_ESTATE, "patch setup needs the host mesh");
    const int npatch = (int)((n_el + kPatch - 1) / kPatch);
    const bool by_length = npe == 8 || (npe == 10 && long_elements(ctx->h_conn, ctx->h_X, n_el, npe));
    const std::vector<int32_t> perm = morton_order(ctx->h_conn, ctx->h_X, n_el, npe, by_length);
    std::vector<int32_t> epos(n_el);
    for (int64_t k = 0; k < n_el; ++k) epos[perm[k]] = (int32_t)k;
    hipStream_t s = ctx->stream;
    const int64_t ngfr = (int64_t)ctx->ngf * GF, rows = npatch + 1;  // rows of the geometric factors
    struct Scratch {  // element positions, first slots, sizes, results; waits before the host vectors go
        jfm_ctx *ctx;
        int32_t *p = nullptr, *node = nullptr;
        ~Scratch() {
            (void)hipStreamSynchronize(ctx->stream);
            jfm_free(ctx, p);
            jfm_free(ctx, node);
        }
    } tmp{ctx};
    bool done = false;
    struct Release {  // a setup that did not end leaves nothing
        jfm_ctx *ctx;
        bool *done;
        ~Release() {
            if (!*done) jfem_patch_release(ctx);
        }
    } release{ctx, &done};
#define PALLOC(ptr, T, cnt)                                                                 \
    do {                                                                                    \
        ptr = jfm_alloc<T>(ctx, std::max<int64_t>(1, (cnt)));                               \
        if (!ptr) return jfm_fail(ctx, JFM_ENOMEM, "patch operator allocation failed");     \
    } while (0)
    PALLOC(tmp.p, int32_t, n_el + N + kSizes * rows + 8);
    int32_t *d_epos = tmp.p, *first = d_epos + n_el, *sizes = first + N;
    int32_t *out = sizes + kSizes * rows;  // two words, then (aligned) a 64-bit one
    unsigned long long *total = (unsigned long long *)(((uintptr_t)(out + 2) + 7) & ~(uintptr_t)7);
    PALLOC(ctx->eperm, int32_t, n_el);
    PALLOC(ctx->pbase, int32_t, npatch);
    JFM_HIP(ctx, hipMemcpyAsync(ctx->eperm, perm.data(), 4 * n_el, hipMemcpyHostToDevice, s));
    JFM_HIP(ctx, hipMemcpyAsync(d_epos, epos.data(), 4 * n_el, hipMemcpyHostToDevice, s));
    JFM_HIP(ctx, hipMemsetAsync(out, 0, 24, s));
    k_patch_build<false><<<npatch, kPT, 0, s>>>((int)n_el, npe, npatch, ctx->conn, ctx->eperm, d_epos, ctx->inc_ptr, ctx->inc,
                                                sizes, ctx->pbase, out, total, nullptr, nullptr, nullptr, nullptr, nullptr,
                                                nullptr, nullptr, nullptr);
    k_patch_sums<<<kSizes, 1024, 0, s>>>(npatch, sizes);
    int32_t got[2], sum[kSizes];
    unsigned long long lin = 0;
    JFM_HIP(ctx, hipMemcpyAsync(got, out, sizeof got, hipMemcpyDeviceToHost, s));
    JFM_HIP(ctx, hipMemcpyAsync(&lin, total, sizeof lin, hipMemcpyDeviceToHost, s));
    JFM_HIP(ctx, hipMemcpy2DAsync(sum, 4, sizes + npatch, 4 * rows, 4, kSizes, hipMemcpyDeviceToHost, s));
    JFM_HIP(ctx, hipStreamSynchronize(s));
    if (lin > (unsigned long long)INT32_MAX || sum[kNodes] >= INT32_MAX / 3)
        return jfm_fail(ctx, JFM_EINVAL, "patch structure out of range");
    const int64_t npn = sum[kNodes], nb = (int64_t)sum[kShared] + ctx->orphans;
    PALLOC(tmp.node, int32_t, npn);
    PALLOC(ctx->connP, int32_t, npe * n_el);
    PALLOC(ctx->gfP64, double, ngfr * n_el);
    PALLOC(ctx->gfP32, float, ngfr * n_el);
    PALLOC(ctx->pn_ptr, int32_t, rows);
    PALLOC(ctx->pn_cnt, uint16_t, npn);
    PALLOC(ctx->pn_out, int32_t, npn);
    PALLOC(ctx->rstart, int32_t, rows);
    PALLOC(ctx->rbase, int32_t, sum[kRounds]);
    PALLOC(ctx->linT, uint16_t, (int64_t)lin);
    PALLOC(ctx->bptr, int32_t, nb + 1);
    PALLOC(ctx->bnode, int32_t, nb);
    PALLOC(ctx->bpart, double, 3 * (int64_t)sum[kSlots]);
    PALLOC(ctx->ppart, double, npatch);
    // 16-bit connectivity when every patch's ids span at most 65,536
    if (!got[0]) PALLOC(ctx->connP16, uint16_t, npe * n_el);
    // FP32 folded factors: sqrt(cm) invJ, cm = mu w detJ / 5, and lambda / mu
    if (ctx->affine && npe == 10 && ctx->nu_uniform) PALLOC(ctx->gfQ32, float, 9 * n_el);
#undef PALLOC
    ctx->rho32 = (float)(2.0 * ctx->nu0 / (1.0 - 2.0 * ctx->nu0));
    k_patch_build<true><<<npatch, kPT, 0, s>>>((int)n_el, npe, npatch, ctx->conn, ctx->eperm, d_epos, ctx->inc_ptr, ctx->inc,
                                               sizes, ctx->pbase, out, total, ctx->pn_cnt, ctx->pn_out, tmp.node, ctx->rbase,
                                               ctx->linT, first, ctx->bnode, ctx->bptr);
    k_patch_slots<<<(unsigned)((npn + 255) / 256), 256, 0, s>>>((int)npn, tmp.node, first, ctx->pn_out);
    if (ctx->orphans)
        k_patch_orphans<<<1, 1024, 0, s>>>((int)N, ctx->inc_ptr, sum[kSlots], ctx->bnode + sum[kShared], ctx->bptr + sum[kShared]);
    else
        JFM_HIP(ctx, hipMemcpyAsync(ctx->bptr + nb, sizes + kSlots * rows + npatch, 4, hipMemcpyDeviceToDevice, s));
    k_patch_conn<<<(unsigned)((npe * n_el + 255) / 256), 256, 0, s>>>((int)n_el, npe, ctx->eperm, ctx->conn, ctx->pbase, ctx->connP,
                                                                      ctx->connP16);
    JFM_HIP(ctx, hipMemcpyAsync(ctx->pn_ptr, sizes + kNodes * rows, 4 * rows, hipMemcpyDeviceToDevice, s));
    JFM_HIP(ctx, hipMemcpyAsync(ctx->rstart, sizes + kRounds * rows, 4 * rows, hipMemcpyDeviceToDevice, s));
    JFM_HIP(ctx, launch_patch_factors(ctx, ctx->eperm, ctx->gfP64, ctx->gfP32, ctx->gfQ32));
    JFM_HIP(ctx, hipStreamSynchronize(s));
    ctx->npatch = npatch;
    ctx->npn = (int)npn;
    ctx->nbnode = (int)nb;
    ctx->nslot = sum[kSlots];
    ctx->bmaxcnt = got[1];
    ctx->patch_ready = true;
    done = true;
    return JFM_OK;
}

// qsrc for the update kernel of the two-level PCG (nodes in aggregate order)
__global__ __launch_bounds__(256) void k_slot_fill(int N, int32_t *__restrict__ code) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) code[i] = -1;
}

__global__ __launch_bounds__(256) void k_slot_shared(int nb, const int32_t *__restrict__ bptr,
                                                    const int32_t *__restrict__ bnode, int32_t *__restrict__ code) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < nb) code[bnode[b]] = bptr[b] << 5 | (bptr[b + 1] - bptr[b]);
}

__global__ __launch_bounds__(256) void k_slot_gather(int N, const int32_t *__restrict__ agg_nodes,
                                                    const int32_t *__restrict__ code, int32_t *__restrict__ qsrc) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < N) qsrc[k] = code[agg_nodes[k]];
}

bool jfem_patch_defer_shared(const jfm_ctx *ctx, int op) {
    static const bool on = [] {
        const char *v = std::getenv("JFEM_DEFER_SHARED");
        return !(v && v[0] == '0');
    }();
    // the patch kernel's dot must be the element energies (nothing left for
    // the shared nodes), its partials final (one per patch)
    return on && op == JFM_OP_MATFREE && jfem_patch_form(ctx, op) && ctx->affine && ctx->npe == 10 &&
           ctx->npatch <= kMaxPart && ctx->qsrc && ctx->qsrc_gen == ctx->coarse_gen;
}

int jfem_patch_qsrc(jfm_ctx *ctx) {
    if (!ctx->patch_ready || !ctx->agg_nodes || ctx->n_agg == 0) return JFM_OK;
    if (ctx->qsrc && ctx->qsrc_gen == ctx->coarse_gen) return JFM_OK;
    ctx->qsrc_gen = -1;
    // slot codes hold 26 bits of slot index and 5 of count
    if (ctx->bmaxcnt > 31 || ctx->nslot >= (1 << 26)) return JFM_OK;
    const int N = (int)ctx->N;
    if (!ctx->qsrc) ctx->qsrc = jfm_alloc<int32_t>(ctx, std::max(1, N));
    int32_t *code = jfm_alloc<int32_t>(ctx, std::max(1, N));
    if (!ctx->qsrc || !code) {
        jfm_free(ctx, code);
        return jfm_fail(ctx, JFM_ENOMEM, "shared-node code allocation failed");
    }
    hipStream_t s = ctx->stream;
    const unsigned gN = (unsigned)((N + 255) / 256), gB = (unsigned)((ctx->nbnode + 255) / 256);
    k_slot_fill<<<std::max(1u, gN), 256, 0, s>>>(N, code);
    if (ctx->nbnode > 0) k_slot_shared<<<gB, 256, 0, s>>>(ctx->nbnode, ctx->bptr, ctx->bnode, code);
    k_slot_gather<<<std::max(1u, gN), 256, 0, s>>>(N, ctx->agg_nodes, code, ctx->qsrc);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    jfm_free(ctx, code);
    if (e != hipSuccess) return jfm_fail(ctx, JFM_EHIP, std::string("shared-node codes: ") + hipGetErrorString(e));
    ctx->qsrc_gen = ctx->coarse_gen;
    return JFM_OK;
}

// ------------------------------------------------------------- launchers ---
template <typename T> static const T *gfP_of(jfm_ctx *ctx);
template <> const double *gfP_of<double>(jfm_ctx *ctx) { return ctx->gfP64; }
template <> const float *gfP_of<float>(jfm_ctx *ctx) { return ctx->gfP32; }
template <typename T> static const T *keP_of(jfm_ctx *ctx);
template <> const double *keP_of<double>(jfm_ctx *ctx) { return ctx->Ke; }
template <> const float *keP_of<float>(jfm_ctx *ctx) { return ctx->Ke32; }

// Whether the patch kernel forms x.(Kx) from the element energies (no dotv
// reads): the affine Tet10 matrix-free form, with dotv = x, which the PCG
// passes (its directions are zero on fixed DOFs).
// (headline at config 1: 16.10-16.14 ms against 16.26-16.27 ms with the dot
// over the nodes)
template <typename T> static bool energy_dot(const jfm_ctx *ctx, int op, const T *x, const T *dotv) {
    return op == JFM_OP_MATFREE && ctx->affine && ctx->npe == 10 && dotv && dotv == x;
}

// The block partials of the dot go to pout (ctx->ppart when null).
template <int NPE, typename T>
static void patch_kernel(jfm_ctx *ctx, int op, const T *x, T *y, const T *dotv, const int *done, double *pout,
                         T *bpart, int batch) {
    const dim3 grid(xcd_grid(ctx->npatch), batch);
    const int xs = 3 * (int)ctx->N, bs = 3 * ctx->nslot;
    const int n = (int)ctx->n_el;
    double *pp = dotv ? (pout ? pout : ctx->ppart) : nullptr;
    if (energy_dot<T>(ctx, op, x, dotv)) dotv = nullptr;
    auto launch = [&](auto kernel, const T *el, T rho) {
        kernel<<<grid, kPatch, 0, ctx->stream>>>(n, ctx->npatch, ctx->npn, ctx->connP, ctx->connP16, ctx->pbase, el, x,
                                                 ctx->pn_ptr, ctx->pn_cnt,
                                                 ctx->pn_out, ctx->rstart, ctx->rbase, ctx->linT, ctx->fixed, y,
                                                 bpart, dotv, pp, done, rho, xs, bs);
    };
    const bool c16 = ctx->connP16 != nullptr;
    if (op == JFM_OP_EBE) {
        launch(k_ku_patch<NPE, T, true, true, false, false>, keP_of<T>(ctx), T(0));
    } else if (ctx->affine) {
        if constexpr (sizeof(T) == 4 && NPE == 10) {
            if (ctx->gfQ32) {  // folded factors (uniform nu)
                launch(c16 ? k_ku_patch<NPE, T, true, false, true, true> : k_ku_patch<NPE, T, true, false, false, true>,
                       (const T *)ctx->gfQ32, (T)ctx->rho32);
                return;
            }
        }
        launch(c16 ? k_ku_patch<NPE, T, true, false, true, false> : k_ku_patch<NPE, T, true, false, false, false>,
               gfP_of<T>(ctx), T(0));
    } else {
        launch(c16 ? k_ku_patch<NPE, T, false, false, true, false> : k_ku_patch<NPE, T, false, false, false, false>,
               gfP_of<T>(ctx), T(0));
    }
}

template <typename T>
static hipError_t patch_phase(jfm_ctx *ctx, int op, const T *x, T *y, const T *dotv, const int *done, double *pout, T *bpart,
                              int batch) {
    if (ctx->n_el == 0) return hipSuccess;
    if (!jfem_patch_form(ctx, op)) return hipErrorInvalidValue;
    switch (ctx->npe) {
    case 10: patch_kernel<10, T>(ctx, op, x, y, dotv, done, pout, bpart, batch); break;
    case 4: patch_kernel<4, T>(ctx, op, x, y, dotv, done, pout, bpart, batch); break;
    case 8: patch_kernel<8, T>(ctx, op, x, y, dotv, done, pout, bpart, batch); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
template <typename T>
hipError_t launch_patch_phase(jfm_ctx *ctx, int op, const T *x, T *y, const T *dotv, const int *done,
                              double *pout) {
    return patch_phase<T>(ctx, op, x, y, dotv, done, pout, (T *)ctx->bpart, 1);
}

template <typename T>
hipError_t launch_patch_combine(jfm_ctx *ctx, T *y, const T *dotv, double *part, const int *done, int *npart) {
    // a multiple of 8 blocks (XCD mapping), one shared node per thread up to
    // kMaxPart blocks (544 at 1.05M DOFs: a second node per thread would
    // double the dependent-load chain of the kernel)
    const int nb = ctx->nbnode;
    const unsigned g = std::min<unsigned>(xcd_grid((unsigned)((std::max(nb, 1) + kBlock - 1) / kBlock)), kMaxPart);
    const int chunk = (int)((nb + g - 1) / g);
    if (npart) *npart = (int)g;
    k_ku_combine<T><<<g, kBlock, 0, ctx->stream>>>(nb, chunk, ctx->bptr, ctx->bnode, (const T *)ctx->bpart,
                                                   ctx->fixed, y, dotv, (ctx->n_el && part) ? ctx->ppart : nullptr,
                                                   ctx->n_el ? ctx->npatch : 0, part, done, 0, 0);
    return hipGetLastError();
}

// y_i = K x_i for `batch` vectors, 3 N values apart, partial sums in bpart
// (3 nslot values each).  A small mesh has fewer patches than the chip has CUs: at
// 27 patches four products in turn took 60 us.
hipError_t launch_patch_batch(jfm_ctx *ctx, const double *x, double *y, double *bpart, int batch) {
    hipError_t e = patch_phase<double>(ctx, JFM_OP_MATFREE, x, y, nullptr, nullptr, nullptr, bpart, batch);
    if (e != hipSuccess || ctx->nbnode == 0) return e;
    const unsigned g = std::min<unsigned>(xcd_grid((unsigned)((ctx->nbnode + kBlock - 1) / kBlock)), kMaxPart);
    const int chunk = (int)((ctx->nbnode + g - 1) / g);
    k_ku_combine<double><<<dim3(g, batch), kBlock, 0, ctx->stream>>>(ctx->nbnode, chunk, ctx->bptr, ctx->bnode, bpart, ctx->fixed, y,
                                                                     nullptr, nullptr, 0, nullptr, nullptr, 3 * (int)ctx->N,
                                                                     3 * ctx->nslot);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_patch_apply(jfm_ctx *ctx, int op, const T *x, T *y, const T *dotv, double *part, const int *done,
                              int *npart) {
    const bool energy = energy_dot<T>(ctx, op, x, dotv);
    if (energy && part && ctx->npatch <= kMaxPart) {
        // the patches' energy partials are the final ones: straight to part,
        // and the shared-node kernel only sums nodes
        hipError_t e = launch_patch_phase<T>(ctx, op, x, y, dotv, done, part);
        if (e != hipSuccess) return e;
        if (npart) *npart = ctx->npatch;
        return launch_patch_combine<T>(ctx, y, nullptr, nullptr, done, nullptr);
    }
    hipError_t e = launch_patch_phase<T>(ctx, op, x, y, dotv, done, nullptr);
    if (e != hipSuccess) return e;
    // with the element energies the shared nodes add nothing to the dot
    return launch_patch_combine<T>(ctx, y, energy ? nullptr : dotv, part, done, npart);
}

template hipError_t launch_patch_phase<double>(jfm_ctx *, int, const double *, double *, const double *, const int *, double *);
template hipError_t launch_patch_phase<float>(jfm_ctx *, int, const float *, float *, const float *, const int *, double *);
template hipError_t launch_patch_combine<double>(jfm_ctx *, double *, const double *, double *, const int *, int *);
template hipError_t launch_patch_combine<float>(jfm_ctx *, float *, const float *, double *, const int *, int *);
template hipError_t launch_patch_apply<double>(jfm_ctx *, int, const double *, double *, const double *, double *, const int *, int *);
template hipError_t launch_patch_apply<float>(jfm_ctx *, int, const float *, float *, const float *, double *, const int *, int *);

}  // namespace jfem
