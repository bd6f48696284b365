// persist.hip -- the whole PCG iteration in one resident kernel (gfx950).
//
// On meshes of up to a few hundred patches an iteration launched kernel by
// kernel is bound by its launches and dependent loads, not by its work: 24 us
// per iteration at 139,587 DOFs (FP64, patch operator, shared nodes, update,
// direction), 11.4 us at 1,575 DOFs; resident they take 11.1 and 3.5 us
// (solves 73.9 -> 33.2 ms and 6.9 -> 2.1 ms).  What is left is latency: at
// 139,587 DOFs 29,000 cycles, of which the element products and nodal sums take
// 5,000, the exchanges 18,000.  Here one workgroup per patch stays
// on its CU for the whole solve.  A patch's node vectors (r, x, z in
// registers, p in LDS), its connectivity and its geometric factors (but a
// Hex8's, which are read from the L2) never leave the CU; what crosses workgroups in an iteration is the partial sums
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
// transfer and reduction in one.  The shared nodes'
// partials are stored first, waited for (vmcnt 0 in every wave, then the block
// barrier), and only then is the scalar published that their readers wait
// for; they move as one or two wide accesses per node, since such accesses
// are not cached and their number is what limits them (as polled 64-bit words
// they took 6.7 us per iteration of 240 workgroups).  Both are reused only in
// the next iteration, whose exchange C a workgroup passes only after every
// other one has read this iteration's.
//
// Progress.  A grid is never larger than the device holds at once, and the
// resident kernels of a process that run together are not either (ResidentHold
// in api.hip), so all workgroups come to run.  Every wait is bounded all the
// same (another process may hold compute units): past the bound a workgroup
// raises the failure flag and returns, the others run into their own bounds,
// and the host repeats the solve with the launched form.  (A cooperative launch
// would be refused while another process has one, and the launched form in its
// place would give other bits.)
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "mf_element.h"
#include "nh_element.h"
#include "persist_exchange.h"

namespace jfem {

// ------------------------------------------------------------------ kernel --
template <typename T> struct PersistArgs {
    int n_el, npatch;
    const uint16_t *connL;    // npe x n_el (patch order): the node's position in its patch
    const T *el;              // geometric factors, patch order
    const double *el64;       // the same in FP64
    T rho;                    // lambda / mu of the folded factors
    int ngf;
    const double *kc;         // heat: conductivities (element order) and the elements' order
    const int32_t *eperm;
    const int32_t *ef, *enext, *fmap;  // heat: the element's first convection face (or -1), the next
    const double *fk;         // one, its element-local nodes (4 bits each) and its matrix
    int nfn;
    const int32_t *pn_n;      // patch nodes: their number; patch p's at kNT p
    const int32_t *pn_node;   // patch node -> node
    const int32_t *pn_slot;   // its partial slot, or -1 (interior)
    const int32_t *pn_sh;     // shared: first slot of its node << 5 | slots
    const uint16_t *pn_cnt;   // its incidences in the patch
    const int32_t *pn_inc;    // their start in lin
    const uint16_t *lin;      // incidences (i, e): i stride + e, ascending e
    const uint8_t *fixed;     // (null: no row mask)
    const T *Minv, *b, *x0, *r0;  // the start and its true residual (null: from 0)
    T *x;                     // (not x0: a solve that gives up leaves the start as it was)
    T *part;                  // the shared nodes' partials, 4 values per slot
    int nslot;
    uint64_t *words;          // the scalars' entries, B and then C
    double rtol2;
    int maxit, polls;
    PcgScalars *S;
    const double *ustate;     // tangent: the displacement it is taken at
    // two-level: per patch node its aggregate; offsets from the aggregates'
    // centroids (per node); the patch's entries, one per aggregate that its
    // owned nodes are in (ce_n[p] of them, at kMaxEntries p: slot in wpart; nodes
    // cn_list[kNT p + cn_ptr[(kMaxEntries + 1) p + e]..]); the
    // aggregates' slots; the coarse operator; exchange words
    const int32_t *pn_agg;
    const T *cd;
    const int32_t *ce_n, *ce_slot, *cn_ptr, *as_ptr;
    const uint16_t *cn_list;
    const float *Ahat;
    int nc, ldc;
    double *wpart;
    uint64_t *zw;
    // systems of one operator side by side: workgroups npatch s .. of the grid
    // solve system s, its b and x ss values further, scalars at S + s
    int64_t ss;
};

// A patch has 512 threads (one node each at most).  The affine Tet10 products
// run on four lanes per element, one per vertex (below), which shortens the
// longest instruction stream of the iteration: with one thread per element and
// three nodes per thread (256 threads) an iteration of a single patch took 7.5
// us, four waves each issuing some 4,300 instructions one after the other.
// 512 threads may hold 256 registers each, enough for a node's and a vertex's
// data; with 256 elements on 1,024 threads the FP64 kernel spilled 73
// registers and an iteration took 9 us.
constexpr int kNT = 512;
template <int NPE> constexpr int persist_elems() { return NPE == 10 ? 128 : (NPE == 8 ? 256 : 512); }

// local node of lane k's slot m: itself, the mid nodes of its edges to
// k ^ 1, k ^ 2, k ^ 3, and those vertices
__host__ __device__ constexpr int tet10_lane_node(int k, int m) {
    constexpr int EDG[4][4] = {{-1, 4, 6, 7}, {4, -1, 5, 8}, {6, 5, -1, 9}, {7, 8, 9, -1}};
    return m == 0 ? k : (m < 4 ? EDG[k][k ^ m] : k ^ (m - 3));
}
template <int D, typename T> __device__ __forceinline__ T quad_xor(T v) {
    return dpp_mov<D == 1 ? kQuadXor1 : (D == 2 ? kQuadXor2 : kQuadXor3)>(v);
}
template <typename T> __device__ __forceinline__ T quad_sum(T v) {
    v += quad_xor<1>(v);
    return v + quad_xor<2>(v);
}
// grad L_j of the vertices j = kv ^ d from invJ: column j - 1, or minus the sum
// of the columns for vertex 0
template <typename T> __device__ __forceinline__ void lane_gradients(const T (&Ji)[9], int kv, T (&g)[9]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int j = kv ^ (d + 1);
#pragma unroll
        for (int b = 0; b < 3; ++b)
            g[3 * d + b] = j == 0 ? -(Ji[b * 3] + Ji[b * 3 + 1] + Ji[b * 3 + 2]) : (j == 1 ? Ji[b * 3] : (j == 2 ? Ji[b * 3 + 1] : Ji[b * 3 + 2]));
    }
}
__device__ __forceinline__ double det_inv(const double (&A)[9]) {
    return A[0] * (A[4] * A[8] - A[5] * A[7]) - A[1] * (A[3] * A[8] - A[5] * A[6]) + A[2] * (A[3] * A[7] - A[4] * A[6]);
}

// An operator of the resident PCG: NC components per node, kLanes lanes per
// element, kIn nodes that a lane reads and kOut that it writes; xc(m, c) is
// component c of p at the lane's m-th node, oc(m, c, v) its term there.
// product() returns the lane's share of p_e.K_e p_e.
template <int N_, int C_, int L_, int I_, int O_, bool D_, int W_> struct OpShape {
    static constexpr int NPE = N_, NC = C_, kLanes = L_, kIn = I_, kOut = O_, kWaves = W_;
    static constexpr bool kDiag = D_;  // diagonal preconditioner (heat, mass)
    static constexpr int kEl = persist_elems<N_>(), kStride = kEl + 1;  // one zero column for padded incidences
    __device__ static int in_node(int kv, int m) { return L_ == 4 && I_ == 7 ? tet10_lane_node(kv, m) : m; }
    template <typename A, typename D, typename X, typename O>
    __device__ static double faces(const A &, const D &, int, const uint16_t *, X &&, O &&) { return 0.0; }
};

// Affine Tet10 elasticity on the four lanes of a quad, lane k holding vertex k.
// With u relative to vertex k, the displacement gradient at vertex k is sum_d
// h_d (x) g_d over the other vertices j = k ^ d, h_d = 4 u_kj - u_j, g_d = grad
// L_j (mf_element.h writes the same sums in the reference frame of vertex 0).
// With sigma_k the stress there (0.2 w detJ folded in), S = sum sigma_k, r_d =
// sigma_k g_d, s_d = S g_d and index 0 the vertex itself (g_0 = -sum g_d):
//     y_corner k = 4 r_0 - s_0,  y_edge kj = 4 ((r_d + r_d of lane j) + (s_0 + s_d)),
// and the element's energy is the sum over its lanes of G_k : (sigma_k + S).
template <typename T_, bool FOLD> struct ElasticTet10 : OpShape<10, 3, 4, 7, 4, false, 2> {
    using T = T_;
    struct Data { T g[9], cl, cm; };
    __device__ static void load(const PersistArgs<T> &A, int k, int kv, bool has, Data &d) {
        T Ji[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) Ji[m] = has ? A.el[(size_t)m * A.n_el + k] : T(0);
        lane_gradients<T>(Ji, kv, d.g);
        d.cl = FOLD ? A.rho : (has ? T(0.2) * A.el[(size_t)9 * A.n_el + k] : T(0));
        d.cm = FOLD ? T(1) : (has ? T(0.2) * A.el[(size_t)10 * A.n_el + k] : T(0));
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<T> &, const Data &D, int, int k, bool has, XC &&xc, OC &&oc) {
        const T *g = D.g, cl = D.cl, cm = D.cm;
        T u0[3], h[3][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) u0[c] = xc(0, c);
#pragma unroll
        for (int d = 0; d < 3; ++d)  // mid node of edge (k, k ^ (d + 1)), vertex k ^ (d + 1)
#pragma unroll
            for (int c = 0; c < 3; ++c) h[d][c] = T(4) * (xc(1 + d, c) - u0[c]) - (xc(4 + d, c) - u0[c]);
        T G[9];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b) G[a * 3 + b] = h[0][a] * g[b] + h[1][a] * g[3 + b] + h[2][a] * g[6 + b];
        const T tr = cl * (G[0] + G[4] + G[8]);
        // 11, 22, 33, 12, 23, 13
        const T s[6] = {tr + T(2) * cm * G[0], tr + T(2) * cm * G[4], tr + T(2) * cm * G[8], cm * (G[1] + G[3]),
                        cm * (G[5] + G[7]), cm * (G[2] + G[6])};
        T S[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) S[m] = quad_sum(s[m]);
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
#pragma unroll
        for (int c = 0; c < 3; ++c) oc(0, c, T(4) * r0[c] - s0[c]);
        auto edge = [&](auto dc) {
            constexpr int d = decltype(dc)::value;
            T r[3], sd[3], f[3];
            mul(s, g + 3 * (d - 1), r);
            mul(S, g + 3 * (d - 1), sd);
#pragma unroll
            for (int c = 0; c < 3; ++c) f[c] = T(4) * ((r[c] + quad_xor<d>(r[c])) + (s0[c] + sd[c]));
            if (k < (k ^ d))  // one of the edge's two lanes
#pragma unroll
                for (int c = 0; c < 3; ++c) oc(d, c, f[c]);
        };
        edge(std::integral_constant<int, 1>{});
        edge(std::integral_constant<int, 2>{});
        edge(std::integral_constant<int, 3>{});
        return has ? (double)en : 0.0;
    }
};

// Neo-Hookean tangent K_T(u) v of an affine Tet10 (nh_element.h), lane k at the
// Gauss point near vertex k (barycentric a there, b elsewhere).  The state (F,
// A = C^-1, S, ln J) is formed once per solve, in FP64, and held in registers.
// With v relative to vertex k, index 0 vertex k and d = 1..3 the vertices k ^ d:
//     grad v = sum_d (c_d - c_0) (x) g_d,  c_0 = 4 b (e_1 + e_2 + e_3),
//     c_d = (4 b - 1) v_d + 4 a e_d + 4 b (the two mid nodes at k ^ d away from k),
// and with P the weighted directional derivative of the first Piola-Kirchhoff
// stress, r_d = P g_d, s_d = (sum of the lanes' P) g_d:
//     y_corner k = (4 b - 1) s_0 + 4 (a - b) r_0,
//     y_edge kj  = 4 (b (s_0 + s_d) + (a - b) (r_d + r_d of lane j)).
template <typename T_> struct TangentTet10 : OpShape<10, 3, 4, 10, 4, false, 2> {
    using T = T_;
    static constexpr double qa = 0.585410196624968, qb = 0.138196601125011;
    // slots 7..9: the mid node of the edge opposite to (k, k ^ d)
    __device__ static int in_node(int kv, int m) {
        constexpr int OPP[10] = {0, 0, 0, 0, 9, 7, 8, 5, 6, 4};  // mid node of the opposite edge
        return m < 7 ? tet10_lane_node(kv, m) : OPP[tet10_lane_node(kv, m - 6)];
    }
    struct Data { T g[9], F[9], A[6], S[6], c1, cl; };  // symmetric ones: 11, 22, 33, 12, 23, 13
    // grad of a nodal field, relative to vertex k
    template <typename U, typename X> __device__ static void gradient(const U (&g)[9], X &&xc, U (&G)[9]) {
        U c[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const U v0 = xc(0, i);
            const U e1 = xc(1, i) - v0, e2 = xc(2, i) - v0, e3 = xc(3, i) - v0;
            const U f1 = xc(7, i) - v0, f2 = xc(8, i) - v0, f3 = xc(9, i) - v0;
            const U c0 = U(4 * qb) * (e1 + e2 + e3);
            c[0][i] = U(4 * qb - 1) * (xc(4, i) - v0) + U(4 * qa) * e1 + U(4 * qb) * (f2 + f3) - c0;
            c[1][i] = U(4 * qb - 1) * (xc(5, i) - v0) + U(4 * qa) * e2 + U(4 * qb) * (f1 + f3) - c0;
            c[2][i] = U(4 * qb - 1) * (xc(6, i) - v0) + U(4 * qa) * e3 + U(4 * qb) * (f1 + f2) - c0;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int b = 0; b < 3; ++b) G[i * 3 + b] = c[0][i] * g[b] + c[1][i] * g[3 + b] + c[2][i] * g[6 + b];
    }
    __device__ static void load(const PersistArgs<T> &A, int k, int kv, bool has, Data &d) {
        double Ji[9], g[9], H[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) Ji[m] = has ? A.el64[(size_t)m * A.n_el + k] : (m % 4 == 0 ? 1.0 : 0.0);
        lane_gradients<double>(Ji, kv, g);
        const double cl = has ? A.el64[(size_t)9 * A.n_el + k] : 0.0, cm = has ? A.el64[(size_t)10 * A.n_el + k] : 0.0;
        const int lb = kNT * (k / kEl);
        gradient<double>(g, [&](int m, int c) -> double {
            return has ? A.ustate[3 * (size_t)A.pn_node[lb + A.connL[(size_t)in_node(kv, m) * A.n_el + k]] + c] : 0.0;
        }, H);
        const double I[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
        double F[9], C[9], S[9], lnJ;
        nh_state<double>(H, I, cl, cm, F, C, S, lnJ);  // H is the physical gradient already
#pragma unroll
        for (int m = 0; m < 9; ++m) {
            d.g[m] = (T)g[m];
            d.F[m] = (T)F[m];
        }
        constexpr int ix[6] = {0, 4, 8, 1, 5, 2};
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            d.A[m] = (T)C[ix[m]];
            d.S[m] = (T)S[ix[m]];
        }
        d.c1 = (T)(2.0 * (cm - cl * lnJ));
        d.cl = (T)cl;
    }
    // o = m v for the symmetric m
    __device__ static void mul(const T (&m)[6], const T *v, int stride, T (&o)[3]) {
        const T v0 = v[0], v1 = v[stride], v2 = v[2 * stride];
        o[0] = m[0] * v0 + m[3] * v1 + m[5] * v2;
        o[1] = m[3] * v0 + m[1] * v1 + m[4] * v2;
        o[2] = m[5] * v0 + m[4] * v1 + m[2] * v2;
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<T> &, const Data &D, int, int k, bool has, XC &&xc, OC &&oc) {
        T G[9], P[9];
        gradient<T>(D.g, xc, G);
        // dE = sym(F' G), AdE = A dE, dS = c1 AdE A + cl tr(AdE) A, P = G S + F dS
        T E[6];
        auto fg = [&](int a, int b) -> T { return D.F[a] * G[b] + D.F[3 + a] * G[3 + b] + D.F[6 + a] * G[6 + b]; };
        E[0] = fg(0, 0);
        E[1] = fg(1, 1);
        E[2] = fg(2, 2);
        E[3] = T(0.5) * (fg(0, 1) + fg(1, 0));
        E[4] = T(0.5) * (fg(1, 2) + fg(2, 1));
        E[5] = T(0.5) * (fg(0, 2) + fg(2, 0));
        const T Ec[9] = {E[0], E[3], E[5], E[3], E[1], E[4], E[5], E[4], E[2]};
        T B[9];  // A dE, row-major
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            T o[3];
            mul(D.A, Ec + b, 3, o);
#pragma unroll
            for (int a = 0; a < 3; ++a) B[a * 3 + b] = o[a];
        }
        const T tr = D.cl * (B[0] + B[4] + B[8]);
        T dS[6];
        auto ba = [&](int a, int b) -> T {  // (A dE A)_ab
            constexpr int ix[9] = {0, 3, 5, 3, 1, 4, 5, 4, 2};
            return B[a * 3] * D.A[ix[b]] + B[a * 3 + 1] * D.A[ix[3 + b]] + B[a * 3 + 2] * D.A[ix[6 + b]];
        };
        dS[0] = D.c1 * ba(0, 0) + tr * D.A[0];
        dS[1] = D.c1 * ba(1, 1) + tr * D.A[1];
        dS[2] = D.c1 * ba(2, 2) + tr * D.A[2];
        dS[3] = D.c1 * ba(0, 1) + tr * D.A[3];
        dS[4] = D.c1 * ba(1, 2) + tr * D.A[4];
        dS[5] = D.c1 * ba(0, 2) + tr * D.A[5];
        T en = T(0);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            T u[3], w[3];
            mul(D.S, G + 3 * a, 1, u);     // row a of G S
            mul(dS, D.F + 3 * a, 1, w);    // row a of F dS
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                P[a * 3 + b] = u[b] + w[b];
                en += G[a * 3 + b] * P[a * 3 + b];
            }
        }
        T Q[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) Q[m] = quad_sum(P[m]);
        const T *g = D.g;
        T g0[3], s0[3], r0[3];
#pragma unroll
        for (int b = 0; b < 3; ++b) g0[b] = -(g[b] + g[3 + b] + g[6 + b]);
        auto app = [&](const T (&M)[9], const T *v, T (&o)[3]) {
#pragma unroll
            for (int a = 0; a < 3; ++a) o[a] = M[a * 3] * v[0] + M[a * 3 + 1] * v[1] + M[a * 3 + 2] * v[2];
        };
        app(Q, g0, s0);
        app(P, g0, r0);
#pragma unroll
        for (int c = 0; c < 3; ++c) oc(0, c, T(4 * qb - 1) * s0[c] + T(4 * (qa - qb)) * r0[c]);
        auto edge = [&](auto dc) {
            constexpr int d = decltype(dc)::value;
            T r[3], sd[3], f[3];
            app(P, g + 3 * (d - 1), r);
            app(Q, g + 3 * (d - 1), sd);
#pragma unroll
            for (int c = 0; c < 3; ++c) f[c] = T(4 * (qa - qb)) * (r[c] + quad_xor<d>(r[c])) + T(4 * qb) * (s0[c] + sd[c]);
            if (k < (k ^ d))
#pragma unroll
                for (int c = 0; c < 3; ++c) oc(d, c, f[c]);
        };
        edge(std::integral_constant<int, 1>{});
        edge(std::integral_constant<int, 2>{});
        edge(std::integral_constant<int, 3>{});
        return has ? (double)en : 0.0;
    }
};

// Hex8 elasticity (2 x 2 x 2 Gauss points) on two lanes per element, lane k with
// the four nodes and the four points of one face zeta = -+1.  Lane 1 works in the
// frame mirrored in zeta: its node m is node m ^ 4, its derivatives along zeta
// change sign, and both lanes run the same code.  Gradients are formed from the
// edges' differences, so translations drop out exactly; in the end the lanes swap
// their terms of the other's nodes.  (One lane per element would hold 72 values
// of gradients, or idle half of the threads.)
template <typename T_> struct ElasticHex8 : OpShape<8, 3, 2, 8, 4, false, 2> {
    using T = T_;
    struct Data {};
    __device__ static int in_node(int kv, int m) { return m ^ (4 * kv); }
    __device__ static void load(const PersistArgs<T> &, int, int, bool, Data &) {}
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<T> &A, const Data &, int k, int kv, bool has, XC &&xc, OC &&oc) {
        if (!has) return 0.0;  // both lanes of the element
        constexpr T a0 = T(0.57735026918962576451), dm = T(0.125 * 1.57735026918962576451), dp = T(0.125 * 0.42264973081037423549);
        // the edges' nodes along xi, eta and zeta, ordered by the other two coordinates' signs
        constexpr int E[3][4][2] = {{{0, 1}, {3, 2}, {4, 5}, {7, 6}}, {{0, 3}, {1, 2}, {4, 7}, {5, 6}}, {{0, 4}, {1, 5}, {3, 7}, {2, 6}}};
        const T sg = kv ? T(-1) : T(1);
        T x[8][3], y[8][3];
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                x[i][c] = xc(i, c);
                y[i][c] = T(0);
            }
#pragma unroll 1  // (unrolled, the points' factors would take 88 registers)
        for (int q = 0; q < 4; ++q) {
            const T xi = q & 1 ? a0 : -a0, eta = q & 2 ? a0 : -a0;
            const T am = T(1) - xi, ap = T(1) + xi, bm = T(1) - eta, bp = T(1) + eta;
            const T w[3][4] = {{bm * dm, bp * dm, bm * dp, bp * dp},
                               {am * dm, ap * dm, am * dp, ap * dp},
                               {sg * T(0.125) * am * bm, sg * T(0.125) * ap * bm, sg * T(0.125) * am * bp, sg * T(0.125) * ap * bp}};
            const T *el = A.el + (size_t)((A.ngf > 1 ? q + 4 * kv : 0) * GF) * A.n_el + k;
            T H[9], Ji[9];
#pragma unroll
            for (int m = 0; m < 9; ++m) Ji[m] = el[(size_t)m * A.n_el];
            const T cl = el[(size_t)9 * A.n_el], cm = el[(size_t)10 * A.n_el];
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    T h = T(0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) h += w[c][e] * (x[E[c][e][1]][a] - x[E[c][e][0]][a]);
                    H[3 * a + c] = h;
                }
            T G[9];
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b)
                    G[a * 3 + b] = H[a * 3] * Ji[b * 3] + H[a * 3 + 1] * Ji[b * 3 + 1] + H[a * 3 + 2] * Ji[b * 3 + 2];
            const T tr = cl * (G[0] + G[4] + G[8]);
            const T s01 = cm * (G[1] + G[3]), s02 = cm * (G[2] + G[6]), s12 = cm * (G[5] + G[7]);
            const T s[9] = {tr + T(2) * cm * G[0], s01, s02, s01, tr + T(2) * cm * G[4], s12, s02, s12, tr + T(2) * cm * G[8]};
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const T P = s[a * 3] * Ji[c] + s[a * 3 + 1] * Ji[3 + c] + s[a * 3 + 2] * Ji[6 + c];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const T f = P * w[c][e];
                        y[E[c][e][1]][a] += f;
                        y[E[c][e][0]][a] -= f;
                    }
                }
        }
        double en = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T x0 = kv ? x[4][c] : x[0][c];  // node 0 in both lanes
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const T f = y[m][c] + quad_xor<1>(y[m + 4][c]);
                oc(m, c, f);
                en += (double)(x[m][c] - x0) * (double)f;
            }
        }
        return en;
    }
};

template <typename T_> struct ElasticTet4 : OpShape<4, 3, 1, 4, 4, false, 2> {
    using T = T_;
    struct Data { T f[GF]; };
    __device__ static void load(const PersistArgs<T> &A, int k, int, bool has, Data &d) {
#pragma unroll
        for (int m = 0; m < GF; ++m) d.f[m] = has ? A.el[(size_t)m * A.n_el + k] : T(0);
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<T> &, const Data &D, int, int, bool has, XC &&xc, OC &&oc) {
        double en = 0.0;
        if (has)
            mf_element_f<4, T, true>([&](int, int m) -> T { return D.f[m]; },
                                     [&](int i, T (&v)[3]) { v[0] = xc(i, 0); v[1] = xc(i, 1); v[2] = xc(i, 2); },
                                     [&](int i, T f0, T f1, T f2) {
                                         oc(i, 0, f0);
                                         oc(i, 1, f1);
                                         oc(i, 2, f2);
                                         if (i > 0)  // K_e annihilates translations
                                             en += (double)((xc(i, 0) - xc(0, 0)) * f0 + (xc(i, 1) - xc(0, 1)) * f1 +
                                                            (xc(i, 2) - xc(0, 2)) * f2);
                                     });
        return en;
    }
};

// Conduction (heat.hip), one component.  The convection faces are faces of an
// element each: the element's (first) lane adds their terms to its own.
template <int NPE_, int L_, int I_, int O_> struct HeatShape : OpShape<NPE_, 1, L_, I_, O_, true, 2> {
    using T = double;
    template <typename D, typename X, typename O>
    __device__ static double faces(const PersistArgs<double> &A, const D &d, int k, X &&xe, O &&ye) {
        double en = 0.0;
        for (int f = d.face; f >= 0; f = A.enext[f]) {
            const int map = A.fmap[f];
            const double *K = A.fk + (size_t)f * 36;
            double v[6];
#pragma unroll
            for (int j = 0; j < 6; ++j) v[j] = j < A.nfn ? xe(map >> (4 * j) & 15) : 0.0;
#pragma unroll
            for (int j = 0; j < 6; ++j)
                if (j < A.nfn) {
                    double s = 0.0;
#pragma unroll
                    for (int l = 0; l < 6; ++l) s += K[6 * j + l] * v[l];
                    ye(map >> (4 * j) & 15, s);
                    en += v[j] * s;
                }
        }
        return en;
    }
};
struct HeatTet10 : HeatShape<10, 4, 7, 4> {  // the vertex form of ElasticTet10, sigma = k grad T
    struct Data { double g[9], c; int face; };
    __device__ static void load(const PersistArgs<double> &A, int k, int kv, bool has, Data &d) {
        double Ji[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) Ji[m] = has ? A.el[(size_t)m * A.n_el + k] : (m % 4 == 0 ? 1.0 : 0.0);
        lane_gradients<double>(Ji, kv, d.g);
        d.c = has ? 0.2 * A.kc[A.eperm[k]] * Elem<10>::w(0) / det_inv(Ji) : 0.0;
        d.face = has && kv == 0 && A.ef ? A.ef[k] : -1;
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<double> &, const Data &D, int, int k, bool has, XC &&xc, OC &&oc) {
        const double *g = D.g, u0 = xc(0, 0);
        double h[3], G[3], s[3], S[3], s0 = 0.0, r0 = 0.0, en = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) h[d] = 4.0 * (xc(1 + d, 0) - u0) - (xc(4 + d, 0) - u0);
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            G[b] = h[0] * g[b] + h[1] * g[3 + b] + h[2] * g[6 + b];
            s[b] = D.c * G[b];
            S[b] = quad_sum(s[b]);
            const double g0 = -(g[b] + g[3 + b] + g[6 + b]);
            s0 += S[b] * g0;
            r0 += s[b] * g0;
            en += G[b] * (s[b] + S[b]);
        }
        oc(0, 0, 4.0 * r0 - s0);
        auto edge = [&](auto dc) {
            constexpr int d = decltype(dc)::value;
            const double *gd = g + 3 * (d - 1);
            const double r = s[0] * gd[0] + s[1] * gd[1] + s[2] * gd[2], sd = S[0] * gd[0] + S[1] * gd[1] + S[2] * gd[2];
            const double f = 4.0 * ((r + quad_xor<d>(r)) + (s0 + sd));
            if (k < (k ^ d)) oc(d, 0, f);
        };
        edge(std::integral_constant<int, 1>{});
        edge(std::integral_constant<int, 2>{});
        edge(std::integral_constant<int, 3>{});
        return has ? en : 0.0;
    }
};
template <int NPE_> struct HeatElem : HeatShape<NPE_, 1, NPE_, NPE_> {  // Tet4, Hex8: the Gauss-point form
    struct Data { double kc; int face; };
    __device__ static void load(const PersistArgs<double> &A, int k, int, bool has, Data &d) {
        d.kc = has ? A.kc[A.eperm[k]] : 0.0;
        d.face = has && A.ef ? A.ef[k] : -1;
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<double> &A, const Data &D, int k, int, bool has, XC &&xc, OC &&oc) {
        using EL = Elem<NPE_>;
        if (!has) return 0.0;
        double xe[NPE_], y[NPE_], Ji[9];
        const double x0 = xc(0, 0);
#pragma unroll
        for (int i = 0; i < NPE_; ++i) {
            xe[i] = xc(i, 0) - x0;  // sum grad N = 0
            y[i] = 0.0;
        }
#pragma unroll 1  // (unrolled, the points' factors spill)
        for (int q = 0; q < EL::NGP; ++q) {
            if (q == 0 || A.ngf > 1)
#pragma unroll
                for (int m = 0; m < 9; ++m) Ji[m] = A.el[(size_t)(q * GF + m) * A.n_el + k];
            const double w = D.kc * EL::w(q) / det_inv(Ji);
            double h[3] = {0.0, 0.0, 0.0}, t[3], u[3];
#pragma unroll
            for (int i = 1; i < NPE_; ++i)
#pragma unroll
                for (int c = 0; c < 3; ++c) h[c] += xe[i] * dn_rt<NPE_>(q, i, c);
#pragma unroll
            for (int b = 0; b < 3; ++b) t[b] = w * (Ji[b * 3] * h[0] + Ji[b * 3 + 1] * h[1] + Ji[b * 3 + 2] * h[2]);
#pragma unroll
            for (int c = 0; c < 3; ++c) u[c] = Ji[c] * t[0] + Ji[3 + c] * t[1] + Ji[6 + c] * t[2];
#pragma unroll
            for (int i = 0; i < NPE_; ++i) y[i] += u[0] * dn_rt<NPE_>(q, i, 0) + u[1] * dn_rt<NPE_>(q, i, 1) + u[2] * dn_rt<NPE_>(q, i, 2);
        }
        double en = 0.0;
#pragma unroll
        for (int i = 0; i < NPE_; ++i) {
            oc(i, 0, y[i]);
            en += xe[i] * y[i];
        }
        return en;
    }
};

// Consistent mass of the nodal fit (postprocess.hip), three components.  An
// affine Tet10's is detJ / 2520 times one constant matrix (6 on a corner's
// diagonal, 1 between corners, -4 to the mid nodes at the corner, -6 to the
// others; 32 on a mid node's diagonal, 8 to the opposite one, 16 to the rest),
// applied through the sums over corners (Sc), mid nodes (Se) and the mid nodes
// at a corner (A_i):
//     corner i:  5 x_i + Sc + 2 A_i - 6 Se
//     edge ab:   16 (x_ab + Se) - 8 x_opposite + 2 (x_a + x_b) - 6 Sc
// about 70 operations per component against 36 points of the fit rule.
struct MassTet10 : OpShape<10, 3, 4, 10, 10, true, 4> {  // lanes 0..2: one component each
    using T = double;
    struct Data { double w; };
    __device__ static void load(const PersistArgs<double> &A, int k, int, bool has, Data &d) {
        double Ji[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) Ji[m] = has ? A.el[(size_t)m * A.n_el + k] : (m % 4 == 0 ? 1.0 : 0.0);
        d.w = has ? 1.0 / (2520.0 * det_inv(Ji)) : 0.0;
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<double> &, const Data &D, int, int kv, bool has, XC &&xc, OC &&oc) {
        if (!has || kv == 3) return 0.0;
        double x[10], en = 0.0;
#pragma unroll
        for (int i = 0; i < 10; ++i) x[i] = xc(i, kv);
        const double Sc = (x[0] + x[1]) + (x[2] + x[3]), Se = ((x[4] + x[5]) + (x[6] + x[7])) + (x[8] + x[9]);
        const double At[4] = {x[4] + x[6] + x[7], x[4] + x[5] + x[8], x[5] + x[6] + x[9], x[7] + x[8] + x[9]};
        constexpr int EA[6] = {0, 1, 2, 0, 1, 2}, EB[6] = {1, 2, 0, 3, 3, 3}, EO[6] = {9, 7, 8, 5, 6, 4};
        auto put = [&](int i, double v) {
            const double y = D.w * v;
            oc(i, kv, y);
            en += x[i] * y;
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) put(i, 5.0 * x[i] + Sc + 2.0 * At[i] - 6.0 * Se);
#pragma unroll
        for (int m = 0; m < 6; ++m) put(4 + m, 16.0 * (x[4 + m] + Se) - 8.0 * x[EO[m]] + 2.0 * (x[EA[m]] + x[EB[m]]) - 6.0 * Sc);
        return en;
    }
};
template <int NPE_> struct MassElem : OpShape<NPE_, 3, 1, NPE_, NPE_, true, 2> {  // Tet4, Hex8
    using T = double;
    static constexpr int NW = NPE_ == 8 ? 8 : 1;
    struct Data { double w[NW]; };  // w detJ at the rule's points
    __device__ static void load(const PersistArgs<double> &A, int k, int, bool has, Data &d) {
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            double Ji[9];
#pragma unroll
            for (int m = 0; m < 9; ++m)
                Ji[m] = has ? A.el[(size_t)((A.ngf > 1 ? q : 0) * GF + m) * A.n_el + k] : (m % 4 == 0 ? 1.0 : 0.0);
            d.w[q] = has ? (NPE_ == 8 ? 1.0 : 1.0 / 120.0) / det_inv(Ji) : 0.0;
        }
    }
    template <typename XC, typename OC>
    __device__ static double product(const PersistArgs<double> &, const Data &D, int, int, bool has, XC &&xc, OC &&oc) {
        if (!has) return 0.0;
        double en = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            double x[NPE_], y[NPE_];
#pragma unroll
            for (int i = 0; i < NPE_; ++i) {
                x[i] = xc(i, c);
                y[i] = 0.0;
            }
            if constexpr (NPE_ == 4) {  // detJ / 120 (1 + delta)
                const double s = (x[0] + x[1]) + (x[2] + x[3]);
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = D.w[0] * (s + x[i]);
            } else {
#pragma unroll
                for (int q = 0; q < NW; ++q) {
                    double s = 0.0;
#pragma unroll
                    for (int i = 0; i < NPE_; ++i) s += Elem<NPE_>::N(q, i) * x[i];
                    s *= D.w[q];
#pragma unroll
                    for (int i = 0; i < NPE_; ++i) y[i] += Elem<NPE_>::N(q, i) * s;
                }
            }
#pragma unroll
            for (int i = 0; i < NPE_; ++i) {
                oc(i, c, y[i]);
                en += x[i] * y[i];
            }
        }
        return en;
    }
};

// Most coarse unknowns (kCoarseRows per thread) and aggregates per patch of the
// two-level form.
constexpr int kCoarseRows = 3, kMaxCoarse = kCoarseRows * kNT, kMaxEntries = 64;
template <typename T, bool COARSE> struct CoarseLds {};
template <typename T> struct CoarseLds<T, true> {
    float w[kMaxCoarse], z[kMaxCoarse];  // w = Q' m r (the GEMV's operand, zero padded), zc
    T d[3 * kNT];                        // the nodes' offsets
    float zr[kMaxCoarse];                // the workgroup's rows of zc
    double wz[kNT / 64];
    int start[kMaxEntries + 1], slot[kMaxEntries];
    uint16_t list[kNT];
};

// COARSE: the two-level preconditioner z = M r + m o Q zc, zc = Ahat Q' m r
// (coarse.hip).  The patches' sums of Q' m r go out with exchange C; every
// workgroup then forms w from them, computes its share of the rows of Ahat w,
// and the rows travel as words (16 copies, one per group of workgroups).
template <class Op, bool COARSE>
__global__ __launch_bounds__(kNT, Op::kWaves) void k_pcg_persist(const PersistArgs<typename Op::T> A0) {
    using T = typename Op::T;
    constexpr int NPE = Op::NPE, NC = Op::NC, NL = Op::kLanes, EL = Op::kEl, ST = Op::kStride, NT = kNT, CS = NPE * ST;
    __shared__ T ys[NC * CS];    // element terms: c CS + i ST + element; column EL of row 0 is zero
    __shared__ T ps[NC * NT];    // p at the patch's nodes
    __shared__ GridSumLds<1> shB;
    __shared__ GridSumLds<2> shC;
    __shared__ int bad;
    __shared__ CoarseLds<T, COARSE> co;
    const PersistArgs<T> &A = A0;
    const int nwg = A.npatch, sys = (int)blockIdx.x / nwg, p = (int)blockIdx.x - sys * nwg;
    const int t = (int)threadIdx.x;
    const int el = t / NL, kv = NL > 1 ? t & (NL - 1) : 0;   // its element (and vertex or component)
    const int k = p * EL + el;
    const bool has_el = el < EL && k < A.n_el;
    const int lb = NT * p, nn = A.pn_n[p];
    uint64_t *wordsB = A.words + (size_t)sys * (grid_words(1, nwg) + grid_words(2, nwg)), *wordsC = wordsB + grid_words(1, nwg);
    PcgScalars *S = A.S + sys;
    const Partials<T> part(A.part + (size_t)sys * 4 * A.nslot, A.nslot);
    const T *bvec = A.b + sys * A.ss;
    T *xvec = A.x + sys * A.ss;
    if (t == 0) bad = 0;
    if (t < NC) ys[t * CS + EL] = T(0);

    // the element's data, held for the whole solve
    int cl[Op::kIn], row[Op::kOut];
#pragma unroll
    for (int m = 0; m < Op::kIn; ++m) cl[m] = has_el ? NC * (int)A.connL[(size_t)Op::in_node(kv, m) * A.n_el + k] : 0;
#pragma unroll
    for (int m = 0; m < Op::kOut; ++m) row[m] = Op::in_node(kv, m) * ST + el;
    typename Op::Data data;
    Op::load(A, k, kv, has_el, data);
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
        const uint32_t lo = 2 * m < cnt ? A.lin[base + 2 * m] : (uint32_t)EL;
        const uint32_t hi = 2 * m + 1 < cnt ? A.lin[base + 2 * m + 1] : (uint32_t)EL;
        inc[m] = lo | hi << 16;
    }
    // nodes are sorted by count, most first: the wave's first lane has the most
    const int cw = __builtin_amdgcn_readfirstlane(cnt);
    uint32_t fx = 0;
    T r[NC], z[NC], pv[NC], x[NC];
    constexpr int NM = Op::kDiag ? NC : NC * NC;
    T M[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) M[m] = in ? A.Minv[9 * (size_t)node + (Op::kDiag ? 4 * m : m)] : T(0);
    double bb[1] = {0.0};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const size_t d = 3 * (size_t)node + c;
        if (in && A.fixed && A.fixed[d]) fx |= 1u << c;
        const T bv = in ? bvec[d] : T(0);
        if (own) bb[0] += (double)bv * (double)bv;
        r[c] = in && A.r0 ? A.r0[d] : bv;
        x[c] = in && A.r0 ? A.x0[d] : T(0);
        pv[c] = T(0);
    }
    T dv[3];               // two-level: the node's offset and aggregate
    int agg = 0, ca0[kCoarseRows], ca1[kCoarseRows], ne = 0;
    if constexpr (COARSE) {
        ne = A.ce_n[p];
        agg = in ? 6 * A.pn_agg[lb + t] : 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            dv[c] = in ? A.cd[3 * (size_t)node + c] : T(0);
            co.d[3 * t + c] = dv[c];
        }
        const int32_t *start = A.cn_ptr + (kMaxEntries + 1) * p;
        if (t <= ne) co.start[t] = start[t];
        if (t < ne) co.slot[t] = A.ce_slot[kMaxEntries * p + t];
        if (t < start[ne]) co.list[t] = A.cn_list[lb + t];
#pragma unroll
        for (int j = 0; j < kCoarseRows; ++j) {
            const int i = t + j * NT, g = i / 6;
            ca0[j] = i < A.nc ? A.as_ptr[g] : 0;
            ca1[j] = i < A.nc ? A.as_ptr[g + 1] : 0;
            co.w[i] = 0.0f;
        }
    }
    __syncthreads();  // bad
    uint32_t epoch = 1;
    if (!grid_sum<1, NT>(bb, wordsB, p, nwg, epoch, A.polls, shB, &bad)) {
        if (t == 0) S->fail = 1;
        return;
    }
    const double tol2 = A.rtol2 * bb[0];
    double rz = 0.0, rr = 0.0, rr0 = 0.0, pq = 1.0, alpha_d = 0.0, beta_d = 0.0;
    int it = 0, done = DONE_RUNNING;

    for (;;) {
        // z = M r and the partials of the owned nodes
        double s2[2] = {0.0, 0.0};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if constexpr (Op::kDiag)
                z[c] = M[c] * r[c];
            else
                z[c] = M[3 * c] * r[0] + M[3 * c + 1] * r[1] + M[3 * c + 2] * r[2];
            if (own) {
                s2[0] += (double)r[c] * (double)z[c];
                s2[1] += (double)r[c] * (double)r[c];
            }
        }
        ++epoch;
        if constexpr (COARSE) {
            // the patch's sums of Q' m r per aggregate: [y; d x y], y = m r
            const int lane = t & 63, wv = t >> 6;
#pragma unroll
            for (int c = 0; c < 3; ++c) ps[3 * t + c] = fx >> c & 1u ? T(0) : r[c];
            __syncthreads();
            // a wave per aggregate and half (a patch has owned nodes in three or four)
            for (int u = wv; u < 2 * ne; u += NT / 64) {
                const int e = u >> 1, h = u & 1;
                double w[3] = {0.0, 0.0, 0.0};
                for (int i = co.start[e] + lane; i < co.start[e + 1]; i += 64) {
                    const int l = 3 * (int)co.list[i];
                    const double y0 = ps[l], y1 = ps[l + 1], y2 = ps[l + 2];
                    if (h == 0) {
                        w[0] += y0;
                        w[1] += y1;
                        w[2] += y2;
                    } else {
                        const double d0 = co.d[l], d1 = co.d[l + 1], d2 = co.d[l + 2];
                        w[0] += d1 * y2 - d2 * y1;
                        w[1] += d2 * y0 - d0 * y2;
                        w[2] += d0 * y1 - d1 * y0;
                    }
                }
                double mine = 0.0;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double v = wave_total(w[c]);
                    mine = lane == c ? v : mine;
                }
                if (lane < 3) put_shared(A.wpart + 6 * (size_t)co.slot[e] + 3 * h + lane, mine);
            }
            stores_done();  // before the block barrier in grid_sum, hence before its words
        }
        if (!grid_sum<2, NT>(s2, wordsC, p, nwg, epoch, A.polls, shC, &bad)) break;
        rr = s2[1];
        if (epoch == 2) rr0 = rr;  // the start
        else ++it;
        if (rr <= tol2) {  // the same in every workgroup
            done = DONE_CONVERGED;
            break;
        }
        if constexpr (COARSE) {
            const int lane = t & 63, wv = t >> 6, nc = A.nc;
            double w64[kCoarseRows];
#pragma unroll
            for (int j = 0; j < kCoarseRows; ++j) {
                const int i = t + j * NT, c = i % 6;
                w64[j] = 0.0;
                if (i < nc) {
                    for (int k0 = ca0[j]; k0 < ca1[j]; k0 += 4) {  // four in flight
                        double v[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) v[u] = k0 + u < ca1[j] ? get_shared(A.wpart + 6 * (size_t)(k0 + u) + c) : 0.0;
#pragma unroll
                        for (int u = 0; u < 4; ++u) w64[j] += v[u];
                    }
                    co.w[i] = (float)w64[j];
                }
            }
            __syncthreads();
            uint64_t *zw = A.zw + (size_t)(p / kGroup) * nc;
            const int copies = (nwg + kGroup - 1) / kGroup, ld4 = A.ldc / 4;
            const float4 *w4 = reinterpret_cast<const float4 *>(co.w);
            // this workgroup's rows, stored together: a row at a time from any
            // wave, each line of a copy took eight stores
            const int per = (nc + nwg - 1) / nwg, row0 = p * per, nrow = min(per, nc - row0);
            for (int i = wv; i < nrow; i += NT / 64) {
                const int row = row0 + i;
                const float4 *Ar = reinterpret_cast<const float4 *>(A.Ahat) + (size_t)row * ld4;
                double s = 0.0;
#pragma unroll 4
                for (int q = lane; q < ld4; q += 64) {
                    const float4 a = Ar[q], b = w4[q];
                    s += (double)a.x * b.x + (double)a.y * b.y + (double)a.z * b.z + (double)a.w * b.w;
                }
                const float zr = (float)wave_total(s);
                if (lane == 0) co.zr[i] = zr;
            }
            __syncthreads();
            for (int i = t; i < nrow * copies; i += NT) {
                const int c = i / nrow, k = i - c * nrow;
                put_word(A.zw + (size_t)c * nc + row0 + k, epoch, __float_as_uint(co.zr[k]));
            }
            double wz = 0.0;
#pragma unroll
            for (int j = 0; j < kCoarseRows; ++j) {
                const int i = t + j * NT;
                if (i < nc) {
                    uint32_t bits[1];
                    if (!poll_words<1>(zw + i, 1, epoch, A.polls, bits)) bad = 1;
                    const float zf = __uint_as_float(bits[0]);
                    co.z[i] = zf;
                    wz += w64[j] * (double)zf;
                }
            }
            wz = wave_total(wz);
            if (lane == 0) co.wz[wv] = wz;
            __syncthreads();
            if (bad) break;
#pragma unroll
            for (int q = 0; q < NT / 64; ++q) s2[0] += co.wz[q];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
                const T corr = (T)co.z[agg + c] + (T)co.z[agg + 3 + c1] * dv[c2] - (T)co.z[agg + 3 + c2] * dv[c1];
                z[c] += fx >> c & 1u ? T(0) : corr;
            }
        }
        if (epoch > 2) {
            beta_d = s2[0] / rz;
            if (!(pq > 0.0) || !(s2[0] > 0.0) || !finite(s2[0])) done = DONE_BREAKDOWN;
            else if (it >= A.maxit) done = DONE_MAXIT;
        }
        rz = s2[0];
        if (done) break;
        // p = z + beta p
        const T beta = (T)beta_d;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            pv[c] = z[c] + beta * pv[c];
            ps[NC * t + c] = pv[c];
        }
        __syncthreads();
        // element products; p.Kp as the sum of the elements' energies (p is
        // zero on fixed DOFs)
        double en[1] = {Op::product(
            A, data, k, kv, has_el, [&](int m, int c) -> T { return ps[cl[m] + c]; },
            [&](int m, int c, T v) { ys[c * CS + row[m]] = v; })};
        if constexpr (NC == 1) {
            if (data.face >= 0) {
                wave_sync();  // after the quad's own terms (LDS accesses of one wave stay in order)
                en[0] += Op::faces(
                    A, data, k, [&](int i) -> T { return ps[A.connL[(size_t)i * A.n_el + k]]; },
                    [&](int i, T v) { ys[i * ST + el] += v; });
            }
        }
        __syncthreads();
        // nodal sums in ascending local element order, four incidences' terms
        // in flight at a time
        T q[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) q[c] = T(0);
#pragma unroll
        for (int m0 = 0; m0 < kInc; m0 += 4)
            if (m0 < cw) {  // uniform in the wave
                T v[4][NC];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t w = inc[(m0 + u) / 2];
                    const int m = (int)(u & 1 ? w >> 16 : w & 0xffffu);
#pragma unroll
                    for (int c = 0; c < NC; ++c) v[u][c] = ys[m + c * CS];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int c = 0; c < NC; ++c) q[c] += v[u][c];
            }
        // further incidences: lane by lane, or, where fewer nodes have them than a
        // sixth of the most that one has, node by node with the whole wave (FP64, 72
        // Tet4 around a node: 7.8 us an iteration lane by lane, 4.1 so; 450 of them:
        // 41 and 4.7)
        if (cw > kInc) {  // uniform
            const unsigned long long more = __ballot(cnt > kInc);
            if (6 * __popcll(more) >= cw - kInc)
                for (int m = kInc; m < cnt; ++m) {
                    const int o = (int)A.lin[base + m];
#pragma unroll
                    for (int c = 0; c < NC; ++c) q[c] += ys[o + c * CS];
                }
            else
                for (unsigned long long todo = more; todo; todo &= todo - 1) {
                    const int lane = t & 63, src = __ffsll(todo) - 1;
                    const int b = __builtin_amdgcn_readlane(base, src), n = __builtin_amdgcn_readlane(cnt, src);
                    T s[NC];
#pragma unroll
                    for (int c = 0; c < NC; ++c) s[c] = T(0);
                    for (int m = kInc + lane; m < n; m += 64) {
                        const int o = (int)A.lin[b + m];
#pragma unroll
                        for (int c = 0; c < NC; ++c) s[c] += ys[o + c * CS];
                    }
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        const T all = (T)wave_total((double)s[c]);
                        if (lane == src) q[c] += all;
                    }
                }
        }
        if (slot >= 0) part.template put<NC>(slot, q);
        stores_done();  // before the block barrier in grid_sum, hence before its words
        if (!grid_sum<1, NT>(en, wordsB, p, nwg, epoch, A.polls, shB, &bad)) break;
        pq = en[0];
        alpha_d = (pq > 0.0 && finite(pq)) ? rz / pq : 0.0;
        const T alpha = (T)alpha_d;
        if (slot >= 0) {
            // shared node: all patches' partials in ascending patch order (its
            // own from the registers), the first four in flight together
            constexpr int kS = 4;
            const int n = sh & 31, first = sh >> 5, me = slot - first;
            T v[kS][NC], s[NC];
#pragma unroll
            for (int u = 0; u < kS; ++u) {
#pragma unroll
                for (int c = 0; c < NC; ++c) v[u][c] = u == me ? q[c] : T(0);
                if (u < n && u != me) part.template get<NC>(first + u, v[u]);
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                s[c] = v[0][c];
#pragma unroll
                for (int u = 1; u < kS; ++u) s[c] += v[u][c];
            }
            for (int u = kS; u < n; ++u) {
                T w[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) w[c] = q[c];
                if (u != me) part.template get<NC>(first + u, w);
#pragma unroll
                for (int c = 0; c < NC; ++c) s[c] += w[c];
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) q[c] = s[c];
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (fx >> c & 1u) q[c] = T(0);
            x[c] += alpha * pv[c];
            r[c] -= alpha * q[c];
        }
    }
    if (bad) {
        if (t == 0) S->fail = 1;
        return;
    }
    if (own)
#pragma unroll
        for (int c = 0; c < 3; ++c) xvec[3 * (size_t)node + c] = c < NC ? x[c < NC ? c : 0] : T(0);
    if (p == 0 && t == 0) {
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
__global__ __launch_bounds__(256) void k_persist_clear(int n, uint64_t *__restrict__ words, int nz, uint64_t *__restrict__ zw,
                                                      int nsys, PcgScalars *S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) words[i] = 0;
    if (i < nz) zw[i] = 0;
    if (i < nsys) S[i].fail = 0;
}

// --------------------------------------------------------------- launchers ---
void launch_persist_clear(jfm_ctx *ctx, int n, uint64_t *words, int nz, uint64_t *zw, int nsys, PcgScalars *S) {
    k_persist_clear<<<(std::max(n, nz) + 255) / 256, 256, 0, ctx->stream>>>(n, words, nz, zw, nsys, S);
}

int jfem_persist_workgroups(const jfm_ctx *ctx, int op) { return op == JFM_OP_CSR ? ctx->rows.nwg : ctx->cells.npatch; }

struct PersistLaunch { const void *f = nullptr; PersistGeometry g; };
template <class Op> static PersistLaunch persist_of(bool coarse) {
    const void *f = (const void *)k_pcg_persist<Op, false>;
    if constexpr (!Op::kDiag)
        if (coarse) f = (const void *)k_pcg_persist<Op, true>;
    return {f, {Op::kEl, kNT, Op::kStride}};
}
// the kernel of an operator on this mesh; none: the launched form
template <typename T> static PersistLaunch persist_kernel(const jfm_ctx *ctx, int op, bool coarse) {
    if (coarse && (ctx->nc > kMaxCoarse || ctx->ldc > kMaxCoarse)) return {};
    const bool tet10 = ctx->npe == 10 && ctx->affine;
    if (op == JFM_OP_MATFREE) {
        if constexpr (sizeof(T) == 4)
            if (tet10 && ctx->nu_uniform) return persist_of<ElasticTet10<T, true>>(coarse);
        if (tet10) return persist_of<ElasticTet10<T, false>>(coarse);
        if (ctx->npe == 4) return persist_of<ElasticTet4<T>>(coarse);
        if (ctx->npe == 8) return persist_of<ElasticHex8<T>>(coarse);
    }
    if (op == JFM_OP_TANGENT && tet10) return persist_of<TangentTet10<T>>(coarse);
    if constexpr (sizeof(T) == 8) {
        if (op == kOpHeat) {
            if (tet10) return persist_of<HeatTet10>(coarse);
            if (ctx->npe == 4) return persist_of<HeatElem<4>>(coarse);
            if (ctx->npe == 8) return persist_of<HeatElem<8>>(coarse);
        }
        if (op == kOpMass) {
            if (tet10) return persist_of<MassTet10>(coarse);
            if (ctx->npe == 4) return persist_of<MassElem<4>>(coarse);
            if (ctx->npe == 8) return persist_of<MassElem<8>>(coarse);
        }
    }
    return {};
}

static bool persist_on() {
    static const bool on = [] {
        const char *v = std::getenv("JFEM_PERSIST");
        return !(v && v[0] == '0');
    }();
    return on;
}

template <typename T> bool jfem_persist_maybe(const jfm_ctx *ctx, int op) {
    if (op == JFM_OP_CSR) return persist_on() && !ctx->persist_off && jfem_rows_maybe(ctx);
    if (!persist_on() || ctx->persist_off || !jfem_patch_enabled() || ctx->n_el < 1) return false;
    const PersistLaunch L = persist_kernel<T>(ctx, op, false);
    if (!L.f) return false;
    const int64_t np = (ctx->n_el + L.g.elems - 1) / L.g.elems;
    return np <= kPersistPatches && np <= ctx->cus && (!ctx->cells.ready || ctx->cells.usable);
}

template <typename T> int jfem_persist_ready(jfm_ctx *ctx, int op, int *nsys, bool coarse) {
    // no room for its lists: the launched form, which needs none of them
    auto unless_room = [&](int rc) {
        if (rc != JFM_ENOMEM) return rc;
        ctx->err.clear();
        return (int)JFM_OK;
    };
    const int want = *nsys;
    *nsys = 0;
    if (!jfem_persist_maybe<T>(ctx, op)) return JFM_OK;
    if (op == JFM_OP_CSR) {
        if (coarse) return JFM_OK;
        if (int rc = jfem_rows_setup(ctx)) return unless_room(rc);
        *nsys = ctx->rows.usable ? 1 : 0;
        return JFM_OK;
    }
    const PersistLaunch L = persist_kernel<T>(ctx, op, coarse);
    if (!L.f) return JFM_OK;
    const int64_t np = (ctx->n_el + L.g.elems - 1) / L.g.elems;
    // every workgroup must be resident at once
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, L.f, L.g.threads, 0) != hipSuccess || per_cu < 1) {
        (void)hipGetLastError();
        return JFM_OK;
    }
    if (op == kOpHeat && !ctx->heat_resident) return JFM_OK;
    if (int rc = jfem_cells_setup(ctx, L.g)) return unless_room(rc);
    if (!ctx->cells.usable) return JFM_OK;
    if (coarse) {
        if (int rc = jfem_cells_coarse(ctx, kMaxEntries)) return unless_room(rc);
        if (!ctx->cells.coarse_usable) return JFM_OK;
    }
    int m = want;  // as many systems side by side as fit, a divisor of those asked for
    while (m > 1 && (want % m || m * np > (int64_t)per_cu * ctx->cus)) --m;
    if (int rc = jfem_cells_systems(ctx, m, grid_words(1, (int)np) + grid_words(2, (int)np))) return unless_room(rc);
    *nsys = m;
    return JFM_OK;
}

template <typename T>
hipError_t launch_pcg_persist(jfm_ctx *ctx, int op, const T *Minv, const T *b, const T *x0, const T *r0, T *x, double rtol,
                              int maxit, bool coarse, int nsys, int64_t ss) {
    if (op == JFM_OP_CSR) return launch_pcg_rows<T>(ctx, Minv, b, x0, r0, x, rtol, maxit);
    const auto &C = ctx->cells;
    const PersistLaunch L = persist_kernel<T>(ctx, op, coarse);
    const bool fold = sizeof(T) == 4 && C.gfQ32;
    PersistArgs<T> A{};
    A.n_el = (int)ctx->n_el;
    A.npatch = C.npatch;
    A.connL = C.connL;
    A.el = sizeof(T) == 8 ? (const T *)C.gf64 : (fold ? (const T *)C.gfQ32 : (const T *)C.gf32);
    A.el64 = C.gf64;
    A.rho = fold ? (T)C.rho32 : T(0);
    A.ustate = ctx->ustate64;
    int nz = 0;
    if (coarse) {
        A.pn_agg = C.pn_agg;
        A.cd = sizeof(T) == 8 ? (const T *)ctx->cd64 : (const T *)ctx->cd32;
        A.ce_n = C.ce_n;
        A.ce_slot = C.ce_slot;
        A.cn_ptr = C.cn_ptr;
        A.as_ptr = C.as_ptr;
        A.cn_list = C.cn_list;
        A.Ahat = ctx->Ahat32;
        A.nc = (int)ctx->nc;
        A.ldc = (int)ctx->ldc;
        A.wpart = C.wpart;
        A.zw = C.zw;
        nz = (C.npatch + kGroup - 1) / kGroup * A.nc;
    }
    A.ngf = ctx->ngf;
    A.kc = ctx->heat_k;
    A.eperm = C.eperm;
    if (op == kOpHeat && ctx->hf_h && ctx->hf_n > 0) {
        A.ef = ctx->hf_first;
        A.enext = ctx->hf_next;
        A.fmap = ctx->hf_map;
        A.fk = ctx->hf_K;
        A.nfn = ctx->hf_nfn;
    }
    A.pn_n = C.pn_n;
    A.pn_node = C.pn_node;
    A.pn_slot = C.pn_slot;
    A.pn_sh = C.pn_sh;
    A.pn_cnt = C.pn_cnt;
    A.pn_inc = C.pn_inc;
    A.lin = C.lin;
    A.fixed = op == kOpMass ? nullptr : ctx->fixed;
    A.Minv = Minv;
    A.b = b;
    A.x0 = x0;
    A.r0 = r0;
    A.x = x;
    A.part = (T *)C.part;
    A.nslot = C.nslot;
    A.words = C.words;
    A.rtol2 = rtol * rtol;
    A.maxit = maxit;
    A.polls = ctx->persist_polls;
    A.S = nsys > 1 ? C.S : ctx->S;
    A.ss = ss;
    const int nw = nsys * (grid_words(1, C.npatch) + grid_words(2, C.npatch));
    launch_persist_clear(ctx, nw, C.words, nz, C.zw, nsys, A.S);
    void *args[] = {&A};
    return hipLaunchKernel(L.f, dim3(nsys * C.npatch), dim3(kNT), args, 0, ctx->stream);
}

template bool jfem_persist_maybe<double>(const jfm_ctx *, int);
template bool jfem_persist_maybe<float>(const jfm_ctx *, int);
template int jfem_persist_ready<double>(jfm_ctx *, int, int *, bool);
template int jfem_persist_ready<float>(jfm_ctx *, int, int *, bool);
template hipError_t launch_pcg_persist<double>(jfm_ctx *, int, const double *, const double *, const double *, const double *, double *, double, int, bool, int, int64_t);
template hipError_t launch_pcg_persist<float>(jfm_ctx *, int, const float *, const float *, const float *, const float *, float *, double, int, bool, int, int64_t);

}  // namespace jfem
