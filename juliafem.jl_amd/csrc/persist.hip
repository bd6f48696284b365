// persist.hip -- the whole PCG iteration in one resident kernel (gfx950).
//
// On meshes of up to a few hundred patches an iteration launched kernel by
// kernel is bound by its launches and dependent loads, not by its work: 24 us
// per iteration at 139,587 DOFs (FP64, patch operator, shared nodes, update,
// direction), 11.4 us at 1,575 DOFs; resident they take 13.2 and 3.8 us
// (solves 73.9 -> 39.4 ms and 6.9 -> 2.3 ms).  Here one workgroup per patch stays
// on its CU for the whole solve.  A patch's node vectors (r, x, z in
// registers, p in LDS), its connectivity and its geometric factors never
// leave the CU; what crosses workgroups in an iteration is the partial sums
// of the nodes that patches share and a few scalars:
//
//   z = M r, partials of (r.z, r.r)           -> exchange C: beta, status
//   p = z + beta p in LDS, element products of p into LDS, nodal sums,
//   partials of shared nodes, p.Kp            -> exchange B: alpha
//   shared nodes: the sum of all patches' partials in ascending patch order
//   x += alpha p, r -= alpha q
//
// Every patch keeps its own copy of the vectors at its shared nodes and
// updates it with the same operations in the same order as the other patches
// (same values, same instructions), so nothing but the partials is exchanged
// and the copies stay equal to the bit.  Sums have a fixed order: results are
// reproducible bit for bit, and equal the launched form's up to the order of
// the reductions.
//
// Exchange.  All data that crosses workgroups is stored and loaded past the
// per-XCD L2s (agent scope), and everything else is read-only or private to
// one workgroup, so no cache is flushed or invalidated.  A scalar travels as
// 64-bit words of 32 payload bits and a 32-bit epoch (the iteration): a word
// proves itself current, so one store and one polling load are barrier,
// transfer and reduction in one.  Words of one kind are contiguous over the
// workgroups: a wave's poll is eight 64-byte requests.  The shared nodes'
// partials are stored first, waited for (vmcnt 0 in every wave, then the block
// barrier), and only then is the scalar published that their readers wait
// for; they move as one or two wide accesses per node, since such accesses
// are not cached and their number is what limits them (as polled 64-bit words
// they took 6.7 us per iteration of 240 workgroups).  Both are reused only in
// the next iteration, whose exchange C a workgroup passes only after every
// other one has read this iteration's.
//
// Progress.  The kernel is launched cooperatively, so all its workgroups are
// resident, and every wait is bounded: past the bound a workgroup raises the
// failure flag and returns, the others run into their own bounds, and the
// host repeats the solve with the launched form.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "jfem_device.h"
#include "mf_element.h"

namespace jfem {

// ---------------------------------------------------------------- exchange --
// Polls of one word before a workgroup gives up (each takes at least the
// latency of a load past the L2, about 0.7 us: some seconds in all).
constexpr int kMaxPolls = 1 << 22;

__device__ __forceinline__ void put_word(uint64_t *w, uint32_t epoch, uint32_t bits) {
    __hip_atomic_store(w, (uint64_t)epoch << 32 | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get_word(const uint64_t *w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the payloads of the N words w[i stride] once all of them are of this epoch
template <int N>
__device__ __forceinline__ bool poll_words(const uint64_t *w, int stride, uint32_t epoch, uint32_t (&bits)[N]) {
    for (int k = 0; k < kMaxPolls; ++k) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint64_t v = get_word(w + (size_t)i * stride);
            bits[i] = (uint32_t)v;
            ok = ok && (uint32_t)(v >> 32) == epoch;
        }
        if (ok) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    return false;
}

// A shared node's three values, past the L2: raw buffer accesses with the sc1
// bit (cache policy bit 4).  Slots are 4 T apart.
constexpr int kSc1 = 16;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Partials {
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ Partials(void *p, int slots)
        : rs(__builtin_amdgcn_make_buffer_rsrc(p, 0, slots * 4 * (int)sizeof(T), 0x00027000)) {}
    __device__ __forceinline__ void put(int slot, const T (&v)[3]) const {
        const int o = slot * 4 * (int)sizeof(T);
        if constexpr (sizeof(T) == 8) {
            u32x4 a;
            u32x2 b;
            __builtin_memcpy(&a, v, 16);
            __builtin_memcpy(&b, v + 2, 8);
            __builtin_amdgcn_raw_buffer_store_b128(a, rs, o, 0, kSc1);
            __builtin_amdgcn_raw_buffer_store_b64(b, rs, o + 16, 0, kSc1);
        } else {
            u32x3 a;
            __builtin_memcpy(&a, v, 12);
            __builtin_amdgcn_raw_buffer_store_b96(a, rs, o, 0, kSc1);
        }
    }
    __device__ __forceinline__ void get(int slot, T (&v)[3]) const {
        const int o = slot * 4 * (int)sizeof(T);
        if constexpr (sizeof(T) == 8) {
            const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, kSc1);
            const u32x2 b = __builtin_amdgcn_raw_buffer_load_b64(rs, o + 16, 0, kSc1);
            __builtin_memcpy(v, &a, 16);
            __builtin_memcpy(v + 2, &b, 8);
        } else {
            const u32x3 a = __builtin_amdgcn_raw_buffer_load_b96(rs, o, 0, kSc1);
            __builtin_memcpy(v, &a, 12);
        }
    }
};
// this wave's stores have reached the point where all XCDs see them
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Sum over a wave, in every lane: DPP steps inside the rows of 16 lanes, then
// the four rows in order.  (The LDS-permute butterfly of wave_sum has a
// latency of some 100 cycles per step, and nothing hides it here.)
template <int CTRL> __device__ __forceinline__ double dpp_mov(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0u, (uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0u, (uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
template <int CTRL> __device__ __forceinline__ float dpp_mov(float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), CTRL, 0xf, 0xf, false));
}
constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kQuadXor3 = 0x1b;  // lane ^ 1, 2, 3 of a quad
constexpr int kRowMirror = 0x140, kRowHalfMirror = 0x141;
__device__ __forceinline__ double row_sum(double v) {  // sum of the lane's row of 16
    v += dpp_mov<kQuadXor1>(v);
    v += dpp_mov<kQuadXor2>(v);
    v += dpp_mov<kRowHalfMirror>(v);
    v += dpp_mov<kRowMirror>(v);
    return v;
}
__device__ __forceinline__ double lane_of(double v, int lane) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), lane);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ __forceinline__ double wave_total(double v) {
    v = row_sum(v);
    return (lane_of(v, 0) + lane_of(v, 16)) + (lane_of(v, 32) + lane_of(v, 48));
}

// All-reduce of NV doubles over the workgroups: v in: the thread's share, out:
// the grid's sums, the same bits in every thread of every workgroup; false
// when a wait gave up.  Up to 16 workgroups read each other's words; more form
// groups of 16 (workgroup >> 4) whose first workgroup sums the group's values
// and publishes the sum once per group, and every workgroup reads its group's
// copy of the groups' sums: uncached requests to one line are served one after
// the other, so no line may have more than a few readers.  (240 workgroups
// reading one set of words, or all of them, took 4-6 us per exchange.)  One
// wave polls: lane 16 k + m reads value k of member m, so a sum over members
// is a row sum.  `words` holds 2 NV rows of nwg words, then 16 copies of 2 NV
// rows of 16.  Calls
// that follow each other without a block barrier use different `sh` (a wave
// may still read it when the next one starts).
template <int NV> struct GridSumLds { double a[NV][16], b[NV]; };
constexpr int kGroup = 16;
static_assert(kPersistPatches <= kGroup * kGroup, "two levels");

// the sum over n <= 16 members' words, in every lane of row k (value k)
template <int NV>
__device__ __forceinline__ double sum_members(const uint64_t *words, int stride, int n, uint32_t epoch, int *bad) {
    const int lane = (int)threadIdx.x & 63, k = lane >> 4, m = lane & 15;
    double v = 0.0;
    if (k < NV && m < n) {
        uint32_t bits[2];
        if (!poll_words<2>(words + (size_t)(2 * k) * stride + m, stride, epoch, bits)) *bad = 1;
        v = __longlong_as_double((long long)((uint64_t)bits[1] << 32 | bits[0]));
    }
    return row_sum(v);
}
// lanes 0 and 1 of row k publish its value
template <int NV>
__device__ __forceinline__ void put_rows(uint64_t *words, int stride, int at, uint32_t epoch, double v) {
    const int lane = (int)threadIdx.x & 63, k = lane >> 4, h = lane & 15;
    if (k < NV && h < 2) {
        const uint64_t b = (uint64_t)__double_as_longlong(v);
        put_word(words + (size_t)(2 * k + h) * stride + at, epoch, (uint32_t)(h ? b >> 32 : b));
    }
}

template <int NV, int NT>
__device__ __forceinline__ bool grid_sum(double (&v)[NV], uint64_t *words, int nwg, uint32_t epoch, GridSumLds<NV> &sh,
                                         int *bad) {
    static_assert(NV <= 2 && NT / 64 <= 16, "one row of 16 lanes per value");
    constexpr int kW = NT / 64;
    const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double w = wave_total(v[k]);
        if (lane == 0) sh.a[k][wv] = w;
    }
    __syncthreads();
    if (wv == 0) {
        const int k = lane >> 4, m = lane & 15, wg = (int)blockIdx.x;
        double s = row_sum(k < NV && m < kW ? sh.a[k < NV ? k : 0][m] : 0.0);  // row k: the block's value k
        if (nwg > 1) {
            put_rows<NV>(words, nwg, wg, epoch, s);
            if (nwg > kGroup) {
                uint64_t *top = words + (size_t)(2 * NV) * nwg;
                if (wg % kGroup == 0) {
                    s = sum_members<NV>(words + wg, nwg, min(kGroup, nwg - wg), epoch, bad);
                    // lane 16 r + c: word row r of copy c
                    double mine = 0.0;
#pragma unroll
                    for (int q = 0; q < NV; ++q) {
                        const double vq = lane_of(s, 16 * q);
                        mine = k >> 1 == q ? vq : mine;
                    }
                    const uint64_t b = (uint64_t)__double_as_longlong(mine);
                    if (k < 2 * NV)
                        put_word(top + (size_t)m * (2 * NV * kGroup) + k * kGroup + wg / kGroup, epoch,
                                 (uint32_t)(k & 1 ? b >> 32 : b));
                }
                s = sum_members<NV>(top + (size_t)(wg / kGroup) * (2 * NV * kGroup), kGroup, (nwg + kGroup - 1) / kGroup, epoch, bad);
            } else {
                s = sum_members<NV>(words, nwg, nwg, epoch, bad);
            }
        }
        if (k < NV && m == 0) sh.b[k] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = sh.b[k];
    return *bad == 0;
}

// ------------------------------------------------------------------ kernel --
template <typename T> struct PersistArgs {
    int n_el, npatch;
    const uint16_t *connL;    // npe x n_el (patch order): the node's position in its patch
    const T *el;              // geometric factors, patch order
    T rho;
    const int32_t *pn_ptr;    // patch nodes: range per patch
    const int32_t *pn_node;   // patch node -> node
    const int32_t *pn_slot;   // its partial slot, or -1 (interior)
    const int32_t *pn_sh;     // shared: first slot of its node << 5 | slots
    const uint16_t *pn_cnt;   // its incidences in the patch
    const int32_t *pn_inc;    // their start in lin
    const uint16_t *lin;      // incidences (i, e): 3 i kStride + e, ascending e
    const uint8_t *fixed;
    const T *Minv, *b, *r0;   // r0: the true residual at the x that is given (null: x = 0)
    T *x;
    T *part;                  // the shared nodes' partials, 4 values per slot
    int nslot;
    uint64_t *words;          // the scalars': 2 rows (B), then 4 (C), of npatch + 256
    double rtol2;
    int maxit;
    PcgScalars *S;
};

// A patch's threads and elements.  The affine Tet10 product runs on four
// lanes per element, one per vertex (below), which shortens the longest
// instruction stream of the iteration: with one thread per element and three
// nodes per thread (256 threads) an iteration of a single patch took 7.5 us,
// four waves each issuing some 4,300 instructions one after the other.  512
// threads may hold 256 registers each, enough for a node's and a vertex's
// data; with 256 elements on 1,024 threads the FP64 kernel spilled 73
// registers and an iteration took 9 us.
template <int NPE> struct PersistShape {
    static_assert(NPE == 10 || NPE == 4, "affine Tet10 and Tet4");
    static constexpr bool kVertexLanes = NPE == 10;
    static constexpr int kThreads = 512;  // also the most nodes of a patch
    static constexpr int kEl = kVertexLanes ? kThreads / 4 : kThreads;
    static constexpr int kStride = kEl + 1;                     // one zero column for padded incidences
};

// Affine Tet10 element product on the four lanes of a quad, lane k holding
// vertex k.  With u relative to vertex k, the displacement gradient at vertex
// k is sum_d h_d (x) g_d over the other vertices j = k ^ d, h_d = 4 u_kj - u_j,
// g_d = grad L_j (mf_element.h writes the same sums in the reference frame of
// vertex 0).  With sigma_k the stress there (0.2 w detJ folded in), S = sum
// sigma_k, r_d = sigma_k g_d, s_d = S g_d and index 0 the vertex itself
// (g_0 = -sum g_d):
//     y_corner k = 4 r_0 - s_0,  y_edge kj = 4 ((r_d + r_d of lane j) + (s_0 + s_d)),
// and the element's energy is the sum over its lanes of G_k : (sigma_k + S).
// ex(v, d) returns lane (k ^ d)'s v.
template <typename T, typename XL, typename Out>
__device__ __forceinline__ T tet10_vertex(const T (&g)[9], T cl, T cm, int k, XL &&xl, Out &&out) {
    T u0[3], h[3][3];
    xl(0, u0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        T ue[3], uv[3];
        xl(1 + d, ue);   // mid node of edge (k, k ^ (d + 1))
        xl(4 + d, uv);   // vertex k ^ (d + 1)
#pragma unroll
        for (int c = 0; c < 3; ++c) h[d][c] = T(4) * (ue[c] - u0[c]) - (uv[c] - u0[c]);
    }
    T G[9];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) G[a * 3 + b] = h[0][a] * g[b] + h[1][a] * g[3 + b] + h[2][a] * g[6 + b];
    const T tr = cl * (G[0] + G[4] + G[8]);
    // 11, 22, 33, 12, 23, 13
    T s[6] = {tr + T(2) * cm * G[0], tr + T(2) * cm * G[4], tr + T(2) * cm * G[8], cm * (G[1] + G[3]), cm * (G[5] + G[7]),
              cm * (G[2] + G[6])};
    T S[6];
#pragma unroll
    for (int m = 0; m < 6; ++m) {
        S[m] = s[m] + dpp_mov<kQuadXor1>(s[m]);
        S[m] += dpp_mov<kQuadXor2>(S[m]);
    }
    const T en = G[0] * (s[0] + S[0]) + G[4] * (s[1] + S[1]) + G[8] * (s[2] + S[2]) + (G[1] + G[3]) * (s[3] + S[3]) +
                 (G[5] + G[7]) * (s[4] + S[4]) + (G[2] + G[6]) * (s[5] + S[5]);
    auto mul = [&](const T (&m)[6], const T *v, T (&o)[3]) {
        o[0] = m[0] * v[0] + m[3] * v[1] + m[5] * v[2];
        o[1] = m[3] * v[0] + m[1] * v[1] + m[4] * v[2];
        o[2] = m[5] * v[0] + m[4] * v[1] + m[2] * v[2];
    };
    T g0[3], s0[3], r0[3];
#pragma unroll
    for (int b = 0; b < 3; ++b) g0[b] = -(g[b] + g[3 + b] + g[6 + b]);
    mul(S, g0, s0);
    mul(s, g0, r0);
    out(0, T(4) * r0[0] - s0[0], T(4) * r0[1] - s0[1], T(4) * r0[2] - s0[2]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        T r[3], sd[3], f[3];
        mul(s, g + 3 * d, r);
        mul(S, g + 3 * d, sd);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T o = d == 0 ? dpp_mov<kQuadXor1>(r[c]) : (d == 1 ? dpp_mov<kQuadXor2>(r[c]) : dpp_mov<kQuadXor3>(r[c]));
            f[c] = T(4) * ((r[c] + o) + (s0[c] + sd[c]));
        }
        if (k < (k ^ (d + 1))) out(1 + d, f[0], f[1], f[2]);  // one of the edge's two lanes
    }
    return en;
}

// local node of lane k's slot m: itself, the mid nodes of its edges to
// k ^ 1, k ^ 2, k ^ 3, and those vertices
__host__ __device__ constexpr int tet10_lane_node(int k, int m) {
    constexpr int EDG[4][4] = {{-1, 4, 6, 7}, {4, -1, 5, 8}, {6, 5, -1, 9}, {7, 8, 9, -1}};
    return m == 0 ? k : (m < 4 ? EDG[k][k ^ m] : k ^ (m - 3));
}

template <int NPE, typename T, bool FOLD>
__global__ __launch_bounds__(PersistShape<NPE>::kThreads) void k_pcg_persist(const PersistArgs<T> A) {
    using SH = PersistShape<NPE>;
    constexpr int kPP = SH::kEl, NT = SH::kThreads, ST = SH::kStride;
    constexpr bool VL = SH::kVertexLanes;
    __shared__ T ys[3 * NPE * ST];   // element terms: (3 i + c) ST + element; column kPP is zero
    __shared__ T ps[3 * NT];         // p at the patch's nodes
    __shared__ GridSumLds<1> shB;
    __shared__ GridSumLds<2> shC;
    __shared__ int bad;
    const int t = (int)threadIdx.x, p = (int)blockIdx.x, nwg = A.npatch;
    const int el = VL ? t >> 2 : t, kv = t & 3;   // its element (and vertex)
    const int k = p * kPP + el;
    const bool has_el = el < kPP && k < A.n_el;
    const int lb = A.pn_ptr[p], nn = A.pn_ptr[p + 1] - lb;
    uint64_t *wordsB = A.words, *wordsC = A.words + 2 * (size_t)(nwg + kGroup * kGroup);
    const Partials<T> part(A.part, A.nslot);
    if (t == 0) bad = 0;
    for (int i = t; i < 3 * NPE; i += NT) ys[i * ST + kPP] = T(0);

    // the element's data, held for the whole solve
    constexpr int NC = VL ? 7 : NPE;
    int cl[NC];
    int row[4];   // lane's output rows (vertex lanes)
    constexpr int NF = FOLD ? 9 : GF;
    T fac[NF];
    if constexpr (VL) {
#pragma unroll
        for (int m = 0; m < 7; ++m) {
            const int i = tet10_lane_node(kv, m);
            cl[m] = has_el ? 3 * (int)A.connL[(size_t)i * A.n_el + k] : 0;
            if (m < 4) row[m] = 3 * i * ST + el;
        }
        // grad L_j of the vertices j = kv ^ d from invJ: column j - 1, or
        // minus the sum of the columns for vertex 0
        T Ji[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) Ji[m] = has_el ? A.el[(size_t)m * A.n_el + k] : T(0);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int j = kv ^ (d + 1);
#pragma unroll
            for (int b = 0; b < 3; ++b)
                fac[3 * d + b] = j == 0 ? -(Ji[b * 3] + Ji[b * 3 + 1] + Ji[b * 3 + 2]) : (j == 1 ? Ji[b * 3] : (j == 2 ? Ji[b * 3 + 1] : Ji[b * 3 + 2]));
        }
        if constexpr (!FOLD) {
            fac[9] = has_el ? T(0.2) * A.el[(size_t)9 * A.n_el + k] : T(0);
            fac[10] = has_el ? T(0.2) * A.el[(size_t)10 * A.n_el + k] : T(0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < NPE; ++i) cl[i] = has_el ? 3 * (int)A.connL[(size_t)i * A.n_el + k] : 0;
#pragma unroll
        for (int m = 0; m < NF; ++m) fac[m] = has_el ? A.el[(size_t)m * A.n_el + k] : T(0);
    }
    // the node's data (one node per thread)
    const bool in = t < nn;
    const int cnt = in ? (int)A.pn_cnt[lb + t] : 0, base = in ? A.pn_inc[lb + t] : 0;
    const int slot = in ? A.pn_slot[lb + t] : -1, sh = slot >= 0 ? A.pn_sh[lb + t] : 0;
    const int node = in ? A.pn_node[lb + t] : 0;
    const bool own = in && (slot < 0 || slot == sh >> 5);
    // incidences, padded to the wave's largest count with the zero column
    constexpr int kInc = 24;
    uint32_t inc[kInc / 2];
#pragma unroll
    for (int m = 0; m < kInc / 2; ++m) {
        const uint32_t lo = 2 * m < cnt ? A.lin[base + 2 * m] : (uint32_t)kPP;
        const uint32_t hi = 2 * m + 1 < cnt ? A.lin[base + 2 * m + 1] : (uint32_t)kPP;
        inc[m] = lo | hi << 16;
    }
    // nodes are sorted by count, most first: the wave's first lane has the most
    const int cw = __builtin_amdgcn_readfirstlane(cnt);
    uint32_t fx = 0;
    T r[3], z[3], pv[3], x[3];
    Blk9<T> M;
#pragma unroll
    for (int m = 0; m < 9; ++m) M.v[m] = in ? A.Minv[9 * (size_t)node + m] : T(0);
    double bb[1] = {0.0};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t d = 3 * (size_t)node + c;
        if (in && A.fixed[d]) fx |= 1u << c;
        const T bv = in ? A.b[d] : T(0);
        if (own) bb[0] += (double)bv * (double)bv;
        r[c] = in && A.r0 ? A.r0[d] : bv;
        x[c] = in && A.r0 ? A.x[d] : T(0);
        pv[c] = T(0);
    }
    __syncthreads();  // bad
    uint32_t epoch = 1;
    if (!grid_sum<1, NT>(bb, wordsB, nwg, epoch, shB, &bad)) {
        if (t == 0) A.S->fail = 1;
        return;
    }
    const double tol2 = A.rtol2 * bb[0];
    double rz = 0.0, rr = 0.0, rr0 = 0.0, pq = 1.0, alpha_d = 0.0, beta_d = 0.0;
    int it = 0, done = DONE_RUNNING;

    for (;;) {
        // z = M r and the partials of the owned nodes
        double s2[2] = {0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            z[c] = M.v[3 * c] * r[0] + M.v[3 * c + 1] * r[1] + M.v[3 * c + 2] * r[2];
            if (own) {
                s2[0] += (double)r[c] * (double)z[c];
                s2[1] += (double)r[c] * (double)r[c];
            }
        }
        ++epoch;
        if (!grid_sum<2, NT>(s2, wordsC, nwg, epoch, shC, &bad)) break;
        rr = s2[1];
        if (epoch == 2) {  // the start
            rr0 = rr;
            if (rr <= tol2) done = DONE_CONVERGED;
        } else {
            ++it;
            beta_d = s2[0] / rz;
            if (rr <= tol2) done = DONE_CONVERGED;
            else if (!(pq > 0.0) || !(s2[0] > 0.0) || !finite(s2[0])) done = DONE_BREAKDOWN;
            else if (it >= A.maxit) done = DONE_MAXIT;
        }
        rz = s2[0];
        if (done) break;  // the same in every workgroup
        // p = z + beta p
        const T beta = (T)beta_d;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            pv[c] = z[c] + beta * pv[c];
            ps[3 * t + c] = pv[c];
        }
        __syncthreads();
        // element products; p.Kp as the sum of the elements' energies (p is
        // zero on fixed DOFs and K_e annihilates translations)
        double en[1] = {0.0};
        auto xl = [&](int i, T (&v)[3]) {
            v[0] = ps[cl[i]];
            v[1] = ps[cl[i] + 1];
            v[2] = ps[cl[i] + 2];
        };
        if constexpr (VL) {
            const T cLa = FOLD ? A.rho : fac[NF > 9 ? 9 : 0], cMu = FOLD ? T(1) : fac[NF > 10 ? 10 : 0];
            const T e = tet10_vertex<T>(reinterpret_cast<const T(&)[9]>(fac), cLa, cMu, kv, xl, [&](int m, T f0, T f1, T f2) {
                ys[row[m]] = f0;
                ys[row[m] + ST] = f1;
                ys[row[m] + 2 * ST] = f2;
            });
            if (has_el) en[0] = (double)e;
        } else if (has_el) {
            T x0[3];
            xl(0, x0);
            auto out = [&](int i, T f0, T f1, T f2) {
                ys[(3 * i) * ST + t] = f0;
                ys[(3 * i + 1) * ST + t] = f1;
                ys[(3 * i + 2) * ST + t] = f2;
                if (i > 0) {
                    T v[3];
                    xl(i, v);
                    en[0] += (double)((v[0] - x0[0]) * f0 + (v[1] - x0[1]) * f1 + (v[2] - x0[2]) * f2);
                }
            };
            mf_element_f<NPE, T, true, FOLD>([&](int, int m) -> T { return fac[m]; }, xl, out, A.rho);
        }
        __syncthreads();
        // nodal sums in ascending local element order
        T q[3] = {T(0), T(0), T(0)};
        // four incidences' terms are in flight at a time
#pragma unroll
        for (int m0 = 0; m0 < kInc; m0 += 4)
            if (m0 < cw) {  // uniform in the wave
                T v[4][3];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t w = inc[(m0 + u) / 2];
                    const int m = (int)(u & 1 ? w >> 16 : w & 0xffffu);
#pragma unroll
                    for (int c = 0; c < 3; ++c) v[u][c] = ys[m + c * ST];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int c = 0; c < 3; ++c) q[c] += v[u][c];
            }
        for (int m = kInc; m < cnt; ++m) {
            const int o = (int)A.lin[base + m];
#pragma unroll
            for (int c = 0; c < 3; ++c) q[c] += ys[o + c * ST];
        }
        if (slot >= 0) part.put(slot, q);
        stores_done();  // before the block barrier in grid_sum, hence before its words
        if (!grid_sum<1, NT>(en, wordsB, nwg, epoch, shB, &bad)) break;
        pq = en[0];
        alpha_d = (pq > 0.0 && finite(pq)) ? rz / pq : 0.0;
        const T alpha = (T)alpha_d;
        if (slot >= 0) {
            // shared node: all patches' partials in ascending patch order (its
            // own from the registers), the first four in flight together
            constexpr int kS = 4;
            const int n = sh & 31, first = sh >> 5, me = slot - first;
            T v[kS][3], s[3] = {T(0), T(0), T(0)};
#pragma unroll
            for (int u = 0; u < kS; ++u) {
#pragma unroll
                for (int c = 0; c < 3; ++c) v[u][c] = u == me ? q[c] : T(0);
                if (u < n && u != me) part.get(first + u, v[u]);
            }
#pragma unroll
            for (int u = 0; u < kS; ++u)
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c] += v[u][c];
            for (int u = kS; u < n; ++u) {
                T w[3] = {q[0], q[1], q[2]};
                if (u != me) part.get(first + u, w);
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c] += w[c];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) q[c] = s[c];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (fx >> c & 1u) q[c] = T(0);
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
    if (p == 0 && t == 0) {
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

// no word of an earlier solve is taken for one of this
__global__ __launch_bounds__(256) void k_persist_clear(int n, uint64_t *__restrict__ words, PcgScalars *S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) words[i] = 0;
    if (i == 0) S->fail = 0;
}

// --------------------------------------------------------------- launchers ---
struct PersistLaunch { const void *f = nullptr; PersistGeometry g; };
template <int NPE, typename T, bool FOLD> static PersistLaunch persist_of() {
    using SH = PersistShape<NPE>;
    return {(const void *)k_pcg_persist<NPE, T, FOLD>, {SH::kEl, SH::kThreads, SH::kStride}};
}
template <typename T> static PersistLaunch persist_kernel(const jfm_ctx *ctx) {
    if (ctx->npe == 4) return persist_of<4, T, false>();
    if (ctx->npe != 10 || !ctx->affine) return {};
    if constexpr (sizeof(T) == 4)
        if (ctx->nu_uniform) return persist_of<10, T, true>();
    return persist_of<10, T, false>();
}

template <typename T> int jfem_persist_ready(jfm_ctx *ctx, int op, bool *yes) {
    *yes = false;
    static const bool on = [] {
        const char *v = std::getenv("JFEM_PERSIST");
        return !(v && v[0] == '0');
    }();
    if (!on || ctx->persist_off || op != JFM_OP_MATFREE || !jfem_patch_enabled() || ctx->n_el < 1) return JFM_OK;
    const PersistLaunch L = persist_kernel<T>(ctx);
    if (!L.f) return JFM_OK;
    const int64_t np = (ctx->n_el + L.g.elems - 1) / L.g.elems;
    if (np > kPersistPatches) return JFM_OK;
    // every workgroup must be resident at once
    int per_cu = 0, cus = 0, coop = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, L.f, L.g.threads, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ctx->device) != hipSuccess || !coop ||
        np > (int64_t)per_cu * cus) {
        (void)hipGetLastError();
        return JFM_OK;
    }
    if (int rc = jfem_cells_setup(ctx, L.g)) return rc;
    *yes = ctx->cells.usable;
    return JFM_OK;
}

template <typename T>
hipError_t launch_pcg_persist(jfm_ctx *ctx, const T *Minv, const T *b, const T *r0, T *x, double rtol, int maxit) {
    const auto &C = ctx->cells;
    const PersistLaunch L = persist_kernel<T>(ctx);
    const bool fold = sizeof(T) == 4 && C.gfQ32;
    PersistArgs<T> A{};
    A.n_el = (int)ctx->n_el;
    A.npatch = C.npatch;
    A.connL = C.connL;
    A.el = sizeof(T) == 8 ? (const T *)C.gf64 : (fold ? (const T *)C.gfQ32 : (const T *)C.gf32);
    A.rho = fold ? (T)C.rho32 : T(0);
    A.pn_ptr = C.pn_ptr;
    A.pn_node = C.pn_node;
    A.pn_slot = C.pn_slot;
    A.pn_sh = C.pn_sh;
    A.pn_cnt = C.pn_cnt;
    A.pn_inc = C.pn_inc;
    A.lin = C.lin;
    A.fixed = ctx->fixed;
    A.Minv = Minv;
    A.b = b;
    A.r0 = r0;
    A.x = x;
    A.part = (T *)C.part;
    A.nslot = C.nslot;
    A.words = C.words;
    A.rtol2 = rtol * rtol;
    A.maxit = maxit;
    A.S = ctx->S;
    const int nw = kPersistWords * (C.npatch + kGroup * kGroup);
    k_persist_clear<<<(nw + 255) / 256, 256, 0, ctx->stream>>>(nw, C.words, ctx->S);
    void *args[] = {&A};
    return hipLaunchCooperativeKernel(L.f, dim3(C.npatch), dim3(L.g.threads), args, 0, ctx->stream);
}

template int jfem_persist_ready<double>(jfm_ctx *, int, bool *);
template int jfem_persist_ready<float>(jfm_ctx *, int, bool *);
template hipError_t launch_pcg_persist<double>(jfm_ctx *, const double *, const double *, const double *, double *, double, int);
template hipError_t launch_pcg_persist<float>(jfm_ctx *, const float *, const float *, const float *, float *, double, int);

}  // namespace jfem
