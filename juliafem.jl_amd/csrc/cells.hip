// cells.hip -- the patches of the resident PCG, built on the device (gfx950).
//
// The elements are ordered along a Morton curve of their centroids (on the host:
// a radix sort of 48-bit codes) and cut into patches
// of 128 Tet10, 256 Hex8 or 512 Tet4 elements.  The rest is one workgroup per
// patch: its nodes in the order of their incidence counts (so that the lanes of
// a wave have as many each), each node's incidences in ascending element order,
// and for the nodes that other patches hold too their slots among the partial
// sums, ascending patch.  On the host this took 7.5 ms at 12,810 Tet10 elements;
// the kernels here take 0.13 ms.  No list depends on the order in which threads run.
#include <algorithm>
#include <array>
#include <cmath>
#include <vector>

#include "sort_scan.h"

namespace jfem {

constexpr int kCT = 512;    // threads, and the most nodes of a patch
constexpr int kCK = 2048;   // most incidences of a patch
enum { kCellNodes = 1, kCellShared = 2, kCellEntries = 4 };  // why a mesh does not fit

// One workgroup per patch.  Its incidences sorted by (node, element, local
// node) give the patch's nodes and their incidences; the nodes are then ranked
// by count (most first, then node id).  A node with fewer incidences here than
// in the mesh is shared: from its elements' positions follow the number of its
// patches (pn_sh) and how many of them come before this one (pn_slot).
__global__ __launch_bounds__(kCT) void k_cell_nodes(int n_el, int npe, int ps, int stride, const int32_t *__restrict__ conn,
                                                   const int32_t *__restrict__ perm, const int32_t *__restrict__ epos,
                                                   const int32_t *__restrict__ inc_ptr, const int32_t *__restrict__ inc,
                                                   int32_t *__restrict__ pn_n, int32_t *__restrict__ pn_node,
                                                   uint16_t *__restrict__ pn_cnt, int32_t *__restrict__ pn_inc,
                                                   int32_t *__restrict__ pn_slot, int32_t *__restrict__ pn_sh,
                                                   uint16_t *__restrict__ connL, uint16_t *__restrict__ lin,
                                                   int32_t *__restrict__ psum, int32_t *__restrict__ flags) {
    __shared__ uint64_t key[kCK];
    __shared__ int head[kCT + 1], cnt[kCT], ranked[kCT];
    const int p = blockIdx.x, t = threadIdx.x;
    const int k0 = p * ps, ne = min(ps, n_el - k0), m = ne * npe;
    int n2 = 2;
    while (n2 < m) n2 <<= 1;
    for (int idx = t; idx < n2; idx += kCT) {
        uint64_t v = ~0ull;
        if (idx < m) {
            const int i = idx / ne, kl = idx - i * ne;
            v = (uint64_t)(uint32_t)conn[(size_t)i * n_el + perm[k0 + kl]] << 32 | (uint32_t)(kl << 8 | i);
        }
        key[idx] = v;
    }
    sort_keys<kCT>(key, n2);
    // the nodes, in ascending order: where each one's incidences start
    int first[4], heads = 0, nn;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int idx = 4 * t + j;
        first[j] = idx < m && (idx == 0 || key[idx] >> 32 != key[idx - 1] >> 32);
        heads += first[j];
    }
    int h = block_scan<kCT>(heads, &nn);
    if (nn > kCT) {  // uniform
        if (t == 0) {
            pn_n[p] = 0;
            psum[p] = 0;
            atomicOr(flags, kCellNodes);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (first[j]) head[h++] = 4 * t + j;
    if (t == 0) head[nn] = m;
    __syncthreads();
    const int c = t < nn ? head[t + 1] - head[t] : 0;
    cnt[t] = c;
    __syncthreads();
    int u = 0;  // its rank
    for (int q = 0; q < nn; ++q) u += cnt[q] > c || (cnt[q] == c && q < t);
    if (t < nn) ranked[u] = t;
    __syncthreads();
    // thread t takes the node of rank t
    const int q = t < nn ? ranked[t] : 0, n = t < nn ? cnt[q] : 0, r0 = head[q];
    int all, total, rank;
    const int off = block_scan<kCT>(n, &all);
    const size_t l = (size_t)p * kCT + t;
    const int a = t < nn ? (int)(key[r0] >> 32) : 0;
    const int b0 = t < nn ? inc_ptr[a] : 0, b1 = t < nn ? inc_ptr[a + 1] : 0;
    patches_of_node<kCT>(n < b1 - b0, b0, b1, npe, ps, (n_el + ps - 1) / ps, p, inc, epos, &total, &rank);
    if (total > 31) atomicOr(flags, kCellShared);  // 5 bits
    if (t < nn) {
        const size_t base = (size_t)k0 * npe + off;
        for (int j = 0; j < n; ++j) {
            const uint32_t w = (uint32_t)key[r0 + j];
            const int i = w & 255, kl = (int)(w >> 8);
            lin[base + j] = (uint16_t)(i * stride + kl);
            connL[(size_t)i * n_el + k0 + kl] = (uint16_t)t;
        }
        pn_node[l] = a;
        pn_cnt[l] = (uint16_t)n;
        pn_inc[l] = (int32_t)base;
        pn_slot[l] = rank;
        pn_sh[l] = total;
    }
    int owned;
    (void)block_scan<kCT>(rank == 0 ? total : 0, &owned);
    if (t == 0) {
        pn_n[p] = nn;
        psum[p] = owned;
    }
}

// Each shared node's first slot: in the order of its first patch and rank there.
__global__ __launch_bounds__(kCT) void k_cell_slots(int npatch, const int32_t *__restrict__ pn_n,
                                                   const int32_t *__restrict__ pn_node, const int32_t *__restrict__ pn_slot,
                                                   const int32_t *__restrict__ pn_sh, const int32_t *__restrict__ psum,
                                                   int32_t *__restrict__ first, int32_t *__restrict__ nslot) {
    const int p = blockIdx.x, t = threadIdx.x;
    int before = 0, part;
    for (int q0 = 0; q0 < p; q0 += kCT) {
        (void)block_scan<kCT>(q0 + t < p ? psum[q0 + t] : 0, &part);
        before += part;
    }
    const size_t l = (size_t)p * kCT + t;
    const int n = t < pn_n[p] && pn_slot[l] == 0 ? pn_sh[l] : 0;
    const int o = before + block_scan<kCT>(n, &part);
    if (n) first[pn_node[l]] = o;
    if (p == npatch - 1 && t == 0) *nslot = before + part;
}

// pn_slot: the node's slot of this patch (-1: interior), pn_sh: first slot << 5 | slots
__global__ __launch_bounds__(kCT) void k_cell_final(const int32_t *__restrict__ pn_n, const int32_t *__restrict__ pn_node,
                                                   const int32_t *__restrict__ first, int32_t *__restrict__ pn_slot,
                                                   int32_t *__restrict__ pn_sh) {
    const size_t l = (size_t)blockIdx.x * kCT + threadIdx.x;
    if ((int)threadIdx.x >= pn_n[blockIdx.x] || pn_slot[l] < 0) return;
    const int f = first[pn_node[l]];
    pn_slot[l] += f;
    pn_sh[l] = f << 5 | (pn_sh[l] & 31);
}

// Per patch the aggregates of the nodes it owns (ascending) with those nodes.
__global__ __launch_bounds__(kCT) void k_cell_entries(int n_agg, int max_entries, const int32_t *__restrict__ pn_n,
                                                     const int32_t *__restrict__ pn_node, const int32_t *__restrict__ pn_slot,
                                                     const int32_t *__restrict__ pn_sh, const int32_t *__restrict__ agg,
                                                     int32_t *__restrict__ pn_agg, int32_t *__restrict__ ce_n,
                                                     int32_t *__restrict__ cn_ptr, uint16_t *__restrict__ cn_list,
                                                     int16_t *__restrict__ table, int32_t *__restrict__ flags) {
    __shared__ uint32_t key[kCT];
    const int p = blockIdx.x, t = threadIdx.x;
    const size_t l = (size_t)p * kCT + t;
    uint32_t v = ~0u;
    if (t < pn_n[p]) {
        const int g = agg[pn_node[l]], slot = pn_slot[l];
        pn_agg[l] = g;
        if (slot < 0 || slot == pn_sh[l] >> 5) v = (uint32_t)g << 16 | (uint32_t)t;
    }
    key[t] = v;
    sort_keys<kCT>(key, kCT);
    const uint32_t k = key[t];
    const bool head = k != ~0u && (t == 0 || key[t - 1] >> 16 != k >> 16);
    int ne, nown;
    const int e = block_scan<kCT>(head, &ne);
    (void)block_scan<kCT>(k != ~0u, &nown);
    if (ne > max_entries) {  // uniform
        if (t == 0) {
            ce_n[p] = 0;
            atomicOr(flags, kCellEntries);
        }
        return;
    }
    if (k != ~0u) cn_list[l] = (uint16_t)(k & 0xffff);
    int32_t *start = cn_ptr + (size_t)(max_entries + 1) * p;
    if (head) {
        start[e] = t;
        table[(size_t)p * n_agg + (k >> 16)] = (int16_t)e;
    }
    if (t == 0) {
        start[ne] = nown;
        ce_n[p] = ne;
    }
}

// One workgroup, thread g for aggregate g: its entries' slots, ascending patch.
__global__ __launch_bounds__(kCT) void k_cell_agg_slots(int npatch, int n_agg, int max_entries, const int16_t *__restrict__ table,
                                                       int32_t *__restrict__ as_ptr, int32_t *__restrict__ ce_slot) {
    const int g = threadIdx.x;
    int n = 0, total;
    if (g < n_agg)
#pragma unroll 8
        for (int p = 0; p < npatch; ++p) n += table[(size_t)p * n_agg + g] >= 0;
    int s = block_scan<kCT>(n, &total);
    if (g < n_agg) {
        as_ptr[g] = s;
#pragma unroll 8
        for (int p = 0; p < npatch; ++p) {
            const int e = table[(size_t)p * n_agg + g];
            if (e >= 0) ce_slot[max_entries * p + e] = s++;
        }
    }
    if (g == 0) as_ptr[n_agg] = total;
}

// ------------------------------------------------------------------- host ---
// the bits of v at every third position
static uint64_t spread16(uint64_t v) {
    v &= 0xffff;
    v = (v | v << 16) & 0x0000ff0000ffULL;
    v = (v | v << 8) & 0x00f00f00f00fULL;
    v = (v | v << 4) & 0x0c30c30c30c3ULL;
    v = (v | v << 2) & 0x249249249249ULL;
    return v;
}

// The axes' weights that measure long elements in their own lengths: the least mean
// extent over the axis' own, from some thousand elements; 1 where that is less than
// 1.3 times the least.
static std::array<double, 3> length_weights(const std::vector<int32_t> &conn, const std::vector<double> &X, int64_t n_el, int npe) {
    std::array<double, 3> len = {0.0, 0.0, 0.0}, w;
    const int64_t step = std::max<int64_t>(1, n_el / 1024);
    for (int64_t e = 0; e < n_el; e += step)
        for (int c = 0; c < 3; ++c) {
            double l = 1e300, h = -1e300;
            for (int i = 0; i < npe; ++i) {
                const double x = X[3 * (size_t)conn[e * npe + i] + c];
                l = std::min(l, x);
                h = std::max(h, x);
            }
            len[c] += h - l;
        }
    const double least = std::min({len[0], len[1], len[2]});
    for (int c = 0; c < 3; ++c) w[c] = least > 0.0 && len[c] > 1.3 * least ? least / len[c] : 1.0;
    return w;
}

bool long_elements(const std::vector<int32_t> &conn, const std::vector<double> &X, int64_t n_el, int npe) {
    return length_weights(conn, X, n_el, npe) != std::array<double, 3>{1.0, 1.0, 1.0};
}

// Elements by the Morton code of their centroids, stable in the element id.  One
// scale for the three axes keeps the patches compact: 35% fewer shared-node
// partials than with each axis scaled to the bounding box at 61 x 7 x 5 hexes
// (24,868 against 38,391), and at most 393 nodes a patch instead of 535.  Long
// elements make such patches flat: 40 x 40 x 40 hexes of 10 x 1 x 1 have 133,534
// partials of 480-element patches, and up to 784 nodes in 256 elements, against
// 59,845 and 486 by_length, where an axis counts in element lengths and spans
// 65,536 / 2^k, k the nearest to its length.  (Unrounded, cuts fell across the
// grid's own: 64 x 32 x 32 hexes of 10 x 1 x 1 no longer fitted the resident form,
// 40.4 us an FP64 iteration instead of 22.8, and 480 hexes of 100 x 25 x 26 had up
// to 1,072 nodes, three rounds of threads instead of two.)  Per launched FP64/FP32
// iteration, one scale, bounding box, by_length:
//   Hex8 100 x 25 x 26             38.1/30.2   35.8/28.1   33.9/27.3 us
//   Hex8 128 x 64 x 64, 1 x 1 x 4  178.0/90.4  172.8/84.7  170.0/82.9
//   Tet10 90 x 30 x 30, 10 x 1 x 1 115.2/60.7  101.8/58.5  96.4/57.6
//   Tet10 60 x 20 x 20, 10 x 1 x 1 49.5/32.1   47.6/32.3   46.2/30.6
//   Tet4 100 x 50 x 50, 10 x 1 x 1 77.4/52.4   75.0/57.5   74.9/57.0
// So it is taken by the 480-element patches of Hex8 and of long Tet10, and by the
// resident form where long elements do not fit without.
std::vector<int32_t> morton_order(const std::vector<int32_t> &conn, const std::vector<double> &X, int64_t n_el, int npe, bool by_length) {
    const std::array<double, 3> one = {1.0, 1.0, 1.0}, w = by_length ? length_weights(conn, X, n_el, npe) : one;
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (size_t d = 0; d < X.size(); d += 3)
        for (int c = 0; c < 3; ++c) {
            lo[c] = std::min(lo[c], X[d + c]);
            hi[c] = std::max(hi[c], X[d + c]);
        }
    double side = 0.0, scale[3];
    for (int c = 0; c < 3; ++c) side = std::max(side, w[c] * (hi[c] - lo[c]));
    for (int c = 0; c < 3; ++c) {
        const double l = w[c] * (hi[c] - lo[c]);
        scale[c] = side > 0.0 ? w[c] * (65535.0 / side) : 0.0;
        if (by_length && l * 32768.0 > side) scale[c] = 65535.0 / (hi[c] - lo[c]) * std::exp2(std::round(std::log2(l / side)));
    }
    std::vector<uint64_t> code(n_el);
    for (int64_t e = 0; e < n_el; ++e) {
        double s[3] = {0.0, 0.0, 0.0};
        for (int i = 0; i < npe; ++i)
            for (int c = 0; c < 3; ++c) s[c] += X[3 * (size_t)conn[e * npe + i] + c];
        uint64_t q[3];
        for (int c = 0; c < 3; ++c) q[c] = (uint64_t)std::min(std::max((s[c] / npe - lo[c]) * scale[c], 0.0), 65535.0);
        code[e] = spread16(q[0]) << 2 | spread16(q[1]) << 1 | spread16(q[2]);
    }
    std::vector<int32_t> perm(n_el), next(n_el);
    for (int64_t e = 0; e < n_el; ++e) perm[e] = (int32_t)e;
    for (int shift = 0; shift < 48; shift += 12) {  // least significant digit first
        int32_t start[4097] = {0};
        for (int64_t e = 0; e < n_el; ++e) ++start[(code[e] >> shift & 4095) + 1];
        for (int d = 0; d < 4096; ++d) start[d + 1] += start[d];
        for (int64_t k = 0; k < n_el; ++k) next[start[code[perm[k]] >> shift & 4095]++] = perm[k];
        perm.swap(next);
    }
    return perm;
}

// The resident PCG's patches from the elements' order perm; cells.usable tells
// whether the mesh fits.
static int cells_build(jfm_ctx *ctx, const PersistGeometry &g, const std::vector<int32_t> &perm) {
    auto &C = ctx->cells;
    C.ready = true;
    C.usable = false;
    const int64_t n_el = ctx->n_el, N = ctx->N;
    const int npe = ctx->npe;
    const int64_t np = (n_el + g.elems - 1) / g.elems;
    std::vector<int32_t> epos(n_el);
    for (int64_t k = 0; k < n_el; ++k) epos[perm[k]] = (int32_t)k;
    hipStream_t s = ctx->stream;
    const int64_t pn = np * kCT, rows = (int64_t)ctx->ngf * GF;
    // element positions, first slots of the nodes, sums per patch, flags and slots
    int32_t *tmp = jfm_alloc<int32_t>(ctx, n_el + N + np + 2);
    int32_t *d_epos = tmp, *first = tmp + n_el, *psum = first + N, *out = psum + np;
    const bool fold = ctx->affine && npe == 10 && ctx->nu_uniform;
    bool ok = tmp && (C.eperm = jfm_alloc<int32_t>(ctx, n_el)) && (C.connL = jfm_alloc<uint16_t>(ctx, npe * n_el)) &&
              (C.lin = jfm_alloc<uint16_t>(ctx, npe * n_el)) && (C.pn_n = jfm_alloc<int32_t>(ctx, np)) &&
              (C.pn_node = jfm_alloc<int32_t>(ctx, pn)) && (C.pn_cnt = jfm_alloc<uint16_t>(ctx, pn)) &&
              (C.pn_inc = jfm_alloc<int32_t>(ctx, pn)) && (C.pn_slot = jfm_alloc<int32_t>(ctx, pn)) &&
              (C.pn_sh = jfm_alloc<int32_t>(ctx, pn)) && (C.gf64 = jfm_alloc<double>(ctx, rows * n_el)) &&
              (C.gf32 = jfm_alloc<float>(ctx, rows * n_el)) && (!fold || (C.gfQ32 = jfm_alloc<float>(ctx, 9 * n_el)));
    if (!ok) {
        jfm_free(ctx, tmp);
        jfem_cells_release(ctx);
        return jfm_fail(ctx, JFM_ENOMEM, "resident PCG allocation failed");
    }
    int32_t got[2] = {0, 0};
    hipError_t e = hipMemcpyAsync(C.eperm, perm.data(), 4 * n_el, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(d_epos, epos.data(), 4 * n_el, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemsetAsync(out, 0, 8, s);
    if (e == hipSuccess) {
        k_cell_nodes<<<(unsigned)np, kCT, 0, s>>>((int)n_el, npe, g.elems, g.stride, ctx->conn, C.eperm, d_epos, ctx->inc_ptr,
                                                  ctx->inc, C.pn_n, C.pn_node, C.pn_cnt, C.pn_inc, C.pn_slot, C.pn_sh, C.connL,
                                                  C.lin, psum, out);
        k_cell_slots<<<(unsigned)np, kCT, 0, s>>>((int)np, C.pn_n, C.pn_node, C.pn_slot, C.pn_sh, psum, first, out + 1);
        k_cell_final<<<(unsigned)np, kCT, 0, s>>>(C.pn_n, C.pn_node, first, C.pn_slot, C.pn_sh);
        e = launch_patch_factors(ctx, C.eperm, C.gf64, C.gf32, C.gfQ32);
    }
    if (e == hipSuccess) e = hipMemcpyAsync(got, out, sizeof got, hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);  // also before the host vectors go
    jfm_free(ctx, tmp);
    if (e == hipSuccess) e = w;
    if (e != hipSuccess || got[0] || got[1] >= (1 << 25)) {  // pn_sh holds 26 bits of slot
        jfem_cells_release(ctx);
        C.ready = true;
        return e == hipSuccess ? JFM_OK : jfm_hip_fail(ctx, e, "resident PCG patches");
    }
    C.npatch = (int)np;
    C.nslot = got[1];
    C.epos.swap(epos);
    C.rho32 = (float)(2.0 * ctx->nu0 / (1.0 - 2.0 * ctx->nu0));
    C.usable = true;
    return JFM_OK;
}

// Once per mesh.  Long elements whose patches do not fit are cut again with the
// axes in element lengths.
int jfem_cells_setup(jfm_ctx *ctx, const PersistGeometry &g) {
    auto &C = ctx->cells;
    if (C.ready) return JFM_OK;
    C.ready = true;
    C.usable = false;
    const int64_t n_el = ctx->n_el;
    const int npe = ctx->npe;
    // a node of no element is in no patch; 16-bit incidences
    if (ctx->orphans || g.threads != kCT || g.elems * npe > kCK || npe * g.stride > 65536) return JFM_OK;
    if ((int64_t)ctx->h_conn.size() != n_el * npe || (int64_t)ctx->h_X.size() != 3 * ctx->N) return JFM_OK;
    if (int rc = cells_build(ctx, g, morton_order(ctx->h_conn, ctx->h_X, n_el, npe, false))) return rc;
    if (C.usable || !long_elements(ctx->h_conn, ctx->h_X, n_el, npe)) return JFM_OK;
    return cells_build(ctx, g, morton_order(ctx->h_conn, ctx->h_X, n_el, npe, true));
}

// Per patch the aggregates of its owned nodes, with those nodes, and per
// aggregate the patches' slots (ascending patch), for the current aggregation.
int jfem_cells_coarse(jfm_ctx *ctx, int max_entries) {
    auto &C = ctx->cells;
    if (C.coarse_gen == ctx->coarse_gen) return JFM_OK;
    C.coarse_usable = false;
    for (void **q : {(void **)&C.pn_agg, (void **)&C.ce_n, (void **)&C.ce_slot, (void **)&C.cn_ptr, (void **)&C.as_ptr,
                     (void **)&C.cn_list, (void **)&C.wpart, (void **)&C.zw}) {
        jfm_free(ctx, *q);
        *q = nullptr;
    }
    const int64_t n_agg = ctx->n_agg, np = C.npatch;
    if (!ctx->node_agg || n_agg < 1 || n_agg > kCT) return JFM_OK;
    hipStream_t s = ctx->stream;
    int16_t *table = (int16_t *)jfm_alloc<uint16_t>(ctx, np * n_agg + 4);  // and the flags
    const bool ok = table && (C.pn_agg = jfm_alloc<int32_t>(ctx, np * kCT)) && (C.ce_n = jfm_alloc<int32_t>(ctx, np)) &&
                    (C.ce_slot = jfm_alloc<int32_t>(ctx, np * max_entries)) &&
                    (C.cn_ptr = jfm_alloc<int32_t>(ctx, np * (max_entries + 1))) &&
                    (C.as_ptr = jfm_alloc<int32_t>(ctx, n_agg + 1)) && (C.cn_list = jfm_alloc<uint16_t>(ctx, np * kCT)) &&
                    (C.wpart = jfm_alloc<double>(ctx, 6 * np * max_entries)) &&
                    (C.zw = jfm_alloc<uint64_t>(ctx, 16 * std::max<int64_t>(1, ctx->nc)));
    if (!ok) {
        jfm_free(ctx, table);
        return jfm_fail(ctx, JFM_ENOMEM, "resident PCG allocation failed");
    }
    const int64_t words = (np * n_agg + 1) / 2;  // of 4 bytes; the flags follow
    int32_t *flags = (int32_t *)table + words, got = 0;
    hipError_t e = hipMemsetAsync(table, 0xff, 4 * words, s);
    if (e == hipSuccess) e = hipMemsetAsync(flags, 0, 4, s);
    if (e == hipSuccess) {
        k_cell_entries<<<(unsigned)np, kCT, 0, s>>>((int)n_agg, max_entries, C.pn_n, C.pn_node, C.pn_slot, C.pn_sh, ctx->node_agg,
                                                    C.pn_agg, C.ce_n, C.cn_ptr, C.cn_list, table, flags);
        k_cell_agg_slots<<<1, kCT, 0, s>>>((int)np, (int)n_agg, max_entries, table, C.as_ptr, C.ce_slot);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&got, flags, 4, hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);
    jfm_free(ctx, table);
    if (e == hipSuccess) e = w;
    if (e != hipSuccess) return jfm_hip_fail(ctx, e, "resident PCG coarse lists");
    C.coarse_gen = ctx->coarse_gen;
    C.coarse_usable = got == 0;
    return JFM_OK;
}

int jfem_cells_systems(jfm_ctx *ctx, int m, int words) {
    auto &C = ctx->cells;
    if (m <= C.systems) return JFM_OK;
    for (void *q : {(void *)C.part, (void *)C.words, (void *)C.S}) jfm_free(ctx, q);
    C.systems = 0;
    C.part = jfm_alloc<double>(ctx, (int64_t)m * 4 * std::max(1, C.nslot));
    C.words = jfm_alloc<uint64_t>(ctx, (int64_t)m * words);
    C.S = jfm_alloc<PcgScalars>(ctx, m);
    if (!C.part || !C.words || !C.S) return jfm_fail(ctx, JFM_ENOMEM, "resident PCG allocation failed");
    C.systems = m;
    return JFM_OK;
}

void jfem_cells_release(jfm_ctx *ctx) {
    auto &C = ctx->cells;
    for (void *p : {(void *)C.eperm, (void *)C.connL, (void *)C.pn_n, (void *)C.pn_cnt, (void *)C.pn_node, (void *)C.pn_slot,
                    (void *)C.pn_sh, (void *)C.pn_inc, (void *)C.lin, (void *)C.gf64, (void *)C.gf32,
                    (void *)C.gfQ32, (void *)C.part, (void *)C.words, (void *)C.S, (void *)C.pn_agg, (void *)C.ce_n,
                    (void *)C.ce_slot, (void *)C.cn_ptr, (void *)C.as_ptr, (void *)C.cn_list, (void *)C.wpart, (void *)C.zw})
        jfm_free(ctx, p);
    C = {};
}

}  // namespace jfem
