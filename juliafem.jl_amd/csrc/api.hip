// api.hip -- C ABI of libjfem_hip.so: context, problem upload, assembly,
// operator and solvers.  Declarations and the reference entry point each
// function replaces are in include/jfem.h.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>

#include "jfem_device.h"
#include "jfem_learned.h"

using namespace jfem;

// ================================================================ helpers ==
int jfm_fail(jfm_ctx *ctx, int code, const std::string &msg) {
    if (ctx) ctx->err = msg;
    return code;
}

int jfm_hip_fail(jfm_ctx *ctx, hipError_t e, const char *what) {
    return jfm_fail(ctx, JFM_EHIP, std::string("HIP error ") + hipGetErrorString(e) + " in " + what);
}

template <typename T> T *jfm_alloc(jfm_ctx *ctx, int64_t count) {
    if (count <= 0) count = 1;
    void *p = nullptr;
    const size_t bytes = (size_t)count * sizeof(T);
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    ctx->allocs.push_back(p);
    ctx->bytes += (int64_t)bytes;
    return (T *)p;
}
template uint16_t *jfm_alloc<uint16_t>(jfm_ctx *, int64_t);
template uint64_t *jfm_alloc<uint64_t>(jfm_ctx *, int64_t);

void jfm_free(jfm_ctx *ctx, void *p) {
    if (!p) return;
    auto it = std::find(ctx->allocs.begin(), ctx->allocs.end(), p);
    if (it != ctx->allocs.end()) ctx->allocs.erase(it);
    size_t sz = 0;
    (void)hipMemPtrGetInfo(p, &sz);
    ctx->bytes -= (int64_t)sz;
    (void)hipFree(p);
}

template <typename T> static void free_ptr(jfm_ctx *ctx, T *&p) {
    jfm_free(ctx, (void *)p);
    p = nullptr;
}

#define ALLOC(ctx, ptr, T, n)                                                          \
    do {                                                                               \
        (ptr) = jfm_alloc<T>((ctx), (n));                                              \
        if (!(ptr)) return jfm_fail((ctx), JFM_ENOMEM, "device allocation failed: " #ptr); \
    } while (0)

#define CHECK_LAUNCH(ctx, call)                           \
    do {                                                  \
        hipError_t e_ = (call);                           \
        if (e_ != hipSuccess) return jfm_hip_fail(ctx, e_, #call); \
    } while (0)

// On up to 16 threads with at least `grain` items each: a thread costs some 20 us
// to start.
template <typename F> static void parallel_for(int64_t n, int64_t grain, F f) {
    int nt = (int)std::min<unsigned>(16u, std::max(1u, std::thread::hardware_concurrency()));
    nt = (int)std::min<int64_t>(nt, n / grain);
    if (nt <= 1) {
        f(0, n);
        return;
    }
    std::vector<std::thread> th;
    const int64_t chunk = (n + nt - 1) / nt;
    for (int t = 0; t < nt; ++t) {
        const int64_t a = t * chunk, b = std::min(n, a + chunk);
        if (a >= b) break;
        th.emplace_back([=] { f(a, b); });
    }
    for (auto &x : th) x.join();
}

static void drop_graphs(jfm_ctx *ctx);

static int sync(jfm_ctx *ctx) {
    JFM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return JFM_OK;
}

// ================================================================ context ==
// A resident solve that gave up has waited a second or so, and something else may
// hold the device for longer: the call goes on with launched iterations, and so do
// the next 2^k - 1 calls after k + 1 give-ups in a row.
static void resident_gave_up(jfm_ctx *ctx, int systems) {
    ctx->resident_gave_up += systems;
    ctx->persist_off = true;
    ctx->persist_wait = 1 << std::min(ctx->persist_fails++, 10);
}

// where the calls that solve begin
static void resident_begin(jfm_ctx *ctx) {
    if (ctx->persist_off && --ctx->persist_wait <= 0) ctx->persist_off = false;
    const char *v = std::getenv("JFEM_PERSIST_POLLS");
    ctx->persist_polls = v ? std::min(std::max(std::atoi(v), 0), kMaxPolls) : kMaxPolls;
}

extern "C" int jfm_create(int device, jfm_ctx **out) {
    if (!out) return JFM_EINVAL;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return JFM_EHIP;
    if (device < 0 || device >= ndev) return JFM_EINVAL;
    if (hipSetDevice(device) != hipSuccess) return JFM_EHIP;
    jfm_ctx *ctx = new jfm_ctx();
    ctx->device = device;
    resident_begin(ctx);
    if (hipDeviceGetAttribute(&ctx->cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) ctx->cus = 0;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return JFM_EHIP;
    }
    ctx->S = jfm_alloc<PcgScalars>(ctx, 1);
    if (hipHostMalloc((void **)&ctx->S_host, sizeof(PcgScalars), hipHostMallocDefault) != hipSuccess || !ctx->S) {
        jfm_destroy(ctx);
        return JFM_ENOMEM;
    }
    std::memset(ctx->S_host, 0, sizeof(PcgScalars));
    if (int rc = jfem_noalloc_init(ctx)) {  // device address of the no-allocation entry's scratch
        jfm_destroy(ctx);
        return rc;
    }
    *out = ctx;
    return JFM_OK;
}

extern "C" void jfm_destroy(jfm_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (ctx->stream2) (void)hipStreamSynchronize(ctx->stream2);
    drop_graphs(ctx);
    for (void *p : ctx->allocs) (void)hipFree(p);
    ctx->allocs.clear();
    if (ctx->S_host) (void)hipHostFree(ctx->S_host);
    if (ctx->stream2) {
        (void)hipStreamSynchronize(ctx->stream2);
        (void)hipStreamDestroy(ctx->stream2);
    }
    for (hipEvent_t ev : {ctx->ev_fork, ctx->ev_l0, ctx->ev_l1})
        if (ev) (void)hipEventDestroy(ev);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

extern "C" int jfm_resident_counts(const jfm_ctx *ctx, int64_t *solves, int64_t *gave_up) {
    if (!ctx) return JFM_EINVAL;
    if (solves) *solves = ctx->resident_solves;
    if (gave_up) *gave_up = ctx->resident_gave_up;
    return JFM_OK;
}

extern "C" const char *jfm_last_error(const jfm_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

extern "C" int jfm_get_info(jfm_ctx *ctx, jfm_info *info) {
    if (!ctx || !info) return JFM_EINVAL;
    info->n_nodes = ctx->N;
    info->n_el = ctx->n_el;
    info->n_dofs = ctx->ndof;
    info->nnzb = ctx->nnzb;
    info->nnz = 9 * ctx->nnzb;
    info->n_faces = ctx->n_faces;
    info->npe = ctx->npe;
    info->affine = ctx->affine ? 1 : 0;
    info->device_bytes = ctx->bytes;
    info->n_patches = ctx->patch_ready ? ctx->npatch : 0;
    info->patch_nodes = ctx->patch_ready ? ctx->npn : 0;
    info->shared_nodes = ctx->patch_ready ? ctx->nbnode : 0;
    info->shared_slots = ctx->patch_ready ? ctx->nslot : 0;
    info->patch_conn_bytes = ctx->patch_ready ? (ctx->connP16 ? 2 : 4) : 0;
    info->patch_fp32_factor_rows = ctx->patch_ready ? (ctx->gfQ32 ? 9 : GF) : 0;
    return JFM_OK;
}

// ============================================================ mesh upload ==
static void drop_graphs(jfm_ctx *ctx) {
    for (auto &g : ctx->graphs)
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
    ctx->graphs.clear();
}

static void release_heat(jfm_ctx *ctx) {
    free_ptr(ctx, ctx->heat_k); free_ptr(ctx, ctx->heat_fixed); free_ptr(ctx, ctx->heat_g); free_ptr(ctx, ctx->heat_Minv);
    free_ptr(ctx, ctx->hf_conn); free_ptr(ctx, ctx->hf_ptr); free_ptr(ctx, ctx->hf_inc); free_ptr(ctx, ctx->hf_h);
    free_ptr(ctx, ctx->hf_g); free_ptr(ctx, ctx->hf_text); free_ptr(ctx, ctx->hf_fe);
    free_ptr(ctx, ctx->hf_first); free_ptr(ctx, ctx->hf_next); free_ptr(ctx, ctx->hf_map); free_ptr(ctx, ctx->hf_K);
    ctx->heat_resident = false;
    ctx->hf_n = 0;
    ctx->hf_nfn = 0;
}

static void release_mesh(jfm_ctx *ctx) {
    jfem_learned_drop(ctx);  // no stream2 work may still use the buffers freed here
    free_ptr(ctx, ctx->X); free_ptr(ctx, ctx->conn); free_ptr(ctx, ctx->E); free_ptr(ctx, ctx->nu);
    free_ptr(ctx, ctx->gf64); free_ptr(ctx, ctx->gf32); free_ptr(ctx, ctx->inc_ptr); free_ptr(ctx, ctx->inc);
    free_ptr(ctx, ctx->tl_ws);
    ctx->tl_ws_n = 0;
    free_ptr(ctx, ctx->brow); free_ptr(ctx, ctx->bcol); free_ptr(ctx, ctx->bdiag); free_ptr(ctx, ctx->blk_row);
    free_ptr(ctx, ctx->cptr); free_ptr(ctx, ctx->contrib); free_ptr(ctx, ctx->vals64); free_ptr(ctx, ctx->vals32);
    free_ptr(ctx, ctx->Ke); free_ptr(ctx, ctx->Ke32); free_ptr(ctx, ctx->ye64); free_ptr(ctx, ctx->ye32);
    free_ptr(ctx, ctx->vx64); free_ptr(ctx, ctx->vy64); free_ptr(ctx, ctx->vx32); free_ptr(ctx, ctx->vy32);
    free_ptr(ctx, ctx->fixed); free_ptr(ctx, ctx->g); free_ptr(ctx, ctx->face_conn); free_ptr(ctx, ctx->face_t);
    free_ptr(ctx, ctx->finc_ptr); free_ptr(ctx, ctx->finc); free_ptr(ctx, ctx->fe); free_ptr(ctx, ctx->f_ext);
    free_ptr(ctx, ctx->load); free_ptr(ctx, ctx->u64); free_ptr(ctx, ctx->rr64);
    free_ptr(ctx, ctx->partials); free_ptr(ctx, ctx->counter); free_ptr(ctx, ctx->inc_slot);
    drop_graphs(ctx);
    for (Workspace *w : {&ctx->ws64, &ctx->ws32}) {
        free_ptr(ctx, w->x); free_ptr(ctx, w->r); free_ptr(ctx, w->z); free_ptr(ctx, w->p);
        free_ptr(ctx, w->q); free_ptr(ctx, w->b); free_ptr(ctx, w->Minv);
        w->ok = false;
    }
    free_ptr(ctx, ctx->Mlearn64); free_ptr(ctx, ctx->Mlearn32); free_ptr(ctx, ctx->feat); free_ptr(ctx, ctx->efeat); free_ptr(ctx, ctx->lout);
    free_ptr(ctx, ctx->Muser64); free_ptr(ctx, ctx->Muser32); free_ptr(ctx, ctx->xprobe);
    free_ptr(ctx, ctx->ustate64); free_ptr(ctx, ctx->ustate32); free_ptr(ctx, ctx->Dtan);
    free_ptr(ctx, ctx->nl_u); free_ptr(ctx, ctx->nl_r); free_ptr(ctx, ctx->nl_du); free_ptr(ctx, ctx->nl_zero);
    ctx->has_state = ctx->minv_tangent = false;
    jfem_coarse_release(ctx);
    jfem_patch_release(ctx);
    jfem_cells_release(ctx);
    jfem_rows_release(ctx);
    jfem_train_release(ctx);
    ctx->persist_off = false;
    ctx->persist_wait = ctx->persist_fails = 0;
    release_heat(ctx);
    ctx->h_X.clear();
    ctx->has_user = false;
    ctx->has_mesh = ctx->has_bcs = ctx->assembled = ctx->has_load = false;
    ctx->learned_ready = false;
    ctx->h_conn.clear(); ctx->h_brow.clear(); ctx->h_bcol.clear();
}

extern "C" int jfm_upload_mesh(jfm_ctx *ctx, int64_t n_nodes, const double *X, int64_t n_el, int32_t npe,
                               const int64_t *conn, const double *E, const double *nu, int32_t index_base) {
    if (!ctx) return JFM_EINVAL;
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    if (npe != 10 && npe != 4 && npe != 8)
        return jfm_fail(ctx, JFM_EUNSUPPORTED, "unsupported element: nodes_per_element must be 10 (Tet10), 4 (Tet4) or 8 (Hex8)");
    if (n_nodes <= 0 || n_el < 0 || !X || (n_el > 0 && (!conn || !E || !nu)))
        return jfm_fail(ctx, JFM_EINVAL, "invalid mesh arguments");
    if (index_base != 0 && index_base != 1) return jfm_fail(ctx, JFM_EINVAL, "index_base must be 0 or 1");
    if (n_nodes > (int64_t)INT32_MAX / 3 || n_el * (int64_t)npe * npe > (int64_t)INT32_MAX)
        return jfm_fail(ctx, JFM_EINVAL, "mesh too large for 32-bit indices");
    release_mesh(ctx);
    ctx->N = n_nodes;
    ctx->n_el = n_el;
    ctx->ndof = 3 * n_nodes;
    ctx->npe = npe;
    ctx->ngp = npe == 10 ? 4 : (npe == 4 ? 1 : 8);
    ctx->npair = npe * (npe + 1) / 2;
    ctx->h_X.assign(X, X + 3 * n_nodes);

    // connectivity -> 0-based int32, range checked
    ctx->h_conn.resize((size_t)n_el * npe);
    std::atomic<bool> bad{false};
    parallel_for(n_el * npe, 65536, [&](int64_t a, int64_t b) {
        for (int64_t k = a; k < b; ++k) {
            const int64_t v = conn[k] - index_base;
            if (v < 0 || v >= n_nodes) bad = true;
            ctx->h_conn[k] = (int32_t)v;
        }
    });
    if (bad) return jfm_fail(ctx, JFM_EINVAL, "connectivity references a node outside [base, base+n_nodes)");
    for (int64_t e = 0; e < n_el; ++e)
        if (!(E[e] > 0.0) || !(nu[e] > -1.0 && nu[e] < 0.5))
            return jfm_fail(ctx, JFM_EINVAL, "material out of range (E > 0, -1 < nu < 0.5 required)");
    ctx->nu_uniform = n_el > 0;
    for (int64_t e = 1; e < n_el && ctx->nu_uniform; ++e) ctx->nu_uniform = nu[e] == nu[0];
    ctx->nu0 = n_el > 0 ? nu[0] : 0.0;

    // device copies, incidences and the pattern's sizes (mesh_lists.hip)
    const int64_t n_inc = n_el * npe;
    ALLOC(ctx, ctx->X, double, 3 * n_nodes);
    ALLOC(ctx, ctx->conn, int32_t, n_inc);
    ALLOC(ctx, ctx->E, double, n_el);
    ALLOC(ctx, ctx->nu, double, n_el);
    ALLOC(ctx, ctx->inc_ptr, int32_t, n_nodes + 1);
    ALLOC(ctx, ctx->inc, int32_t, n_inc);
    ALLOC(ctx, ctx->inc_slot, int32_t, n_inc);
    ALLOC(ctx, ctx->brow, int32_t, n_nodes + 1);
    ALLOC(ctx, ctx->bdiag, int32_t, n_nodes);
    ALLOC(ctx, ctx->contrib, int32_t, n_inc * npe);
    struct Scratch {
        jfm_ctx *ctx;
        int32_t *p;
        ~Scratch() { jfm_free(ctx, p); }
    } scratch{ctx, jfm_alloc<int32_t>(ctx, mesh_lists_scratch(n_nodes, n_el, npe))};
    if (!scratch.p) return jfm_fail(ctx, JFM_ENOMEM, "device allocation failed: mesh lists");
    hipStream_t s = ctx->stream;
    JFM_HIP(ctx, hipMemcpyAsync(ctx->X, X, sizeof(double) * 3 * n_nodes, hipMemcpyHostToDevice, s));
    if (n_el > 0) {
        JFM_HIP(ctx, hipMemcpyAsync(ctx->E, E, sizeof(double) * n_el, hipMemcpyHostToDevice, s));
        JFM_HIP(ctx, hipMemcpyAsync(ctx->nu, nu, sizeof(double) * n_el, hipMemcpyHostToDevice, s));
    }
    MeshFlags flags;
    CHECK_LAUNCH(ctx, launch_mesh_lists(ctx, scratch.p, &flags));
    if (flags.large_rows) {
        uint64_t *keys = jfm_alloc<uint64_t>(ctx, 2 * (int64_t)flags.large_entries);
        if (!keys) return jfm_fail(ctx, JFM_ENOMEM, "device allocation failed: mesh lists");
        const hipError_t e = launch_large_rows(ctx, scratch.p, keys, &flags);
        jfm_free(ctx, keys);
        if (e != hipSuccess) return jfm_hip_fail(ctx, e, "large pattern rows");
    }
    const int32_t nnzb = flags.nnzb;
    ctx->nnzb = nnzb;
    ctx->affine = flags.affine;
    ctx->orphans = flags.orphans;
    ctx->ngf = ctx->affine ? 1 : ctx->ngp;
    ALLOC(ctx, ctx->gf64, double, (int64_t)GF * ctx->ngf * n_el);
    ALLOC(ctx, ctx->gf32, float, (int64_t)GF * ctx->ngf * n_el);
    ALLOC(ctx, ctx->bcol, int32_t, nnzb);
    ALLOC(ctx, ctx->blk_row, int32_t, nnzb);
    ALLOC(ctx, ctx->cptr, int32_t, (int64_t)nnzb + 1);
    CHECK_LAUNCH(ctx, launch_pattern_write(ctx, scratch.p));
    ALLOC(ctx, ctx->ye64, double, n_inc * 3);
    ALLOC(ctx, ctx->ye32, float, n_inc * 3);
    ALLOC(ctx, ctx->fixed, uint8_t, 3 * n_nodes);
    ALLOC(ctx, ctx->g, double, 3 * n_nodes);
    ALLOC(ctx, ctx->f_ext, double, 3 * n_nodes);
    ALLOC(ctx, ctx->load, double, 3 * n_nodes);
    ALLOC(ctx, ctx->finc_ptr, int32_t, n_nodes + 1);
    ALLOC(ctx, ctx->vx64, double, 3 * n_nodes);
    ALLOC(ctx, ctx->vy64, double, 3 * n_nodes);
    ALLOC(ctx, ctx->vx32, float, 3 * n_nodes);
    ALLOC(ctx, ctx->vy32, float, 3 * n_nodes);
    ALLOC(ctx, ctx->partials, double, kPartTotal);
    ALLOC(ctx, ctx->counter, unsigned, 64);
    JFM_HIP(ctx, hipMemsetAsync(ctx->fixed, 0, 3 * n_nodes, s));
    JFM_HIP(ctx, hipMemsetAsync(ctx->g, 0, sizeof(double) * 3 * n_nodes, s));
    JFM_HIP(ctx, hipMemsetAsync(ctx->f_ext, 0, sizeof(double) * 3 * n_nodes, s));
    JFM_HIP(ctx, hipMemsetAsync(ctx->load, 0, sizeof(double) * 3 * n_nodes, s));
    JFM_HIP(ctx, hipMemsetAsync(ctx->finc_ptr, 0, sizeof(int32_t) * (n_nodes + 1), s));
    CHECK_LAUNCH(ctx, launch_zero_u32(ctx, ctx->counter, 64));
    int *d_bad = (int *)(ctx->counter + 32);
    CHECK_LAUNCH(ctx, launch_geom_factors(ctx, d_bad));
    int h_bad = 0;
    JFM_HIP(ctx, hipMemcpyAsync(&h_bad, d_bad, sizeof(int), hipMemcpyDeviceToHost, s));
    if (int rc = sync(ctx)) return rc;
    if (h_bad) return jfm_fail(ctx, JFM_ENOTSPD, "element with detJ <= 0 at a Gauss point (inverted or degenerate)");
    // Meshes whose iterations are launched get the patch operator with the upload,
    // so that the products of jfm_apply_noalloc, which may not allocate, take it
    // too.  It needs patches for a good part of the CUs: FP64 Tet10 13.5 against
    // 15.1 us of the two-phase form with 64 of them, 28.1 against 49.6 with 512,
    // curved 15.3 against 14.6 with 51, 15.5 and 15.6 with 63, 15.8 against 17.6 with
    // 82; Hex8 (eight points: more per workgroup) 18.5 against 16.2 with 86, 19.1
    // against 19.9 with 128, 26.1 against 33.0 with 254.  Without room for it (or
    // with indices that do not fit) the mesh is still good for the CSR operator;
    // a failure of the device is one of the upload.
    const int64_t patches = (n_el + kPatchElems - 1) / kPatchElems;
    if (jfem_patch_enabled() && !jfem_persist_maybe<double>(ctx, JFM_OP_MATFREE) && patches >= (npe == 8 ? 192 : 64)) {
        const int rc = jfem_patch_setup(ctx);
        if (rc != JFM_OK && rc != JFM_ENOMEM && rc != JFM_EINVAL) return rc;
        if (rc == JFM_OK) ctx->na_part = jfm_alloc<double>(ctx, 3 * (int64_t)std::max(1, ctx->nslot));
        ctx->patch_upload = ctx->patch_ready && ctx->na_part;
        if (!ctx->patch_upload) {  // all of it or nothing
            jfem_patch_release(ctx);
            ctx->err.clear();
        }
    }
    ctx->has_mesh = true;
    return JFM_OK;
}

// ============================================================ BCs, loads ===
extern "C" int jfm_upload_bcs(jfm_ctx *ctx, const uint8_t *fixed, const double *u_prescribed, int64_t n_faces,
                              int32_t nodes_per_face, const int64_t *face_conn, const double *traction,
                              int32_t index_base) {
    if (!ctx) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "upload the mesh before boundary conditions");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    if (n_faces < 0 || (n_faces > 0 && (!face_conn || !traction)))
        return jfm_fail(ctx, JFM_EINVAL, "invalid face arguments");
    if (n_faces > 0 && nodes_per_face != 6 && nodes_per_face != 3 && nodes_per_face != 4)
        return jfm_fail(ctx, JFM_EUNSUPPORTED, "nodes_per_face must be 6 (Tri6), 3 (Tri3) or 4 (Quad4)");
    const int64_t N = ctx->N, n = ctx->ndof;
    hipStream_t s = ctx->stream;
    if (fixed) JFM_HIP(ctx, hipMemcpyAsync(ctx->fixed, fixed, n, hipMemcpyHostToDevice, s));
    else JFM_HIP(ctx, hipMemsetAsync(ctx->fixed, 0, n, s));
    ctx->g_nonzero = false;
    if (u_prescribed) {
        for (int64_t i = 0; i < n; ++i)
            if (u_prescribed[i] != 0.0 && fixed && fixed[i]) { ctx->g_nonzero = true; break; }
    }
    if (ctx->g_nonzero) {
        std::vector<double> gh(n, 0.0);
        for (int64_t i = 0; i < n; ++i) gh[i] = fixed[i] ? u_prescribed[i] : 0.0;
        JFM_HIP(ctx, hipMemcpyAsync(ctx->g, gh.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        if (int rc = sync(ctx)) return rc;
    } else {
        JFM_HIP(ctx, hipMemsetAsync(ctx->g, 0, sizeof(double) * n, s));
    }
    free_ptr(ctx, ctx->face_conn); free_ptr(ctx, ctx->face_t); free_ptr(ctx, ctx->finc); free_ptr(ctx, ctx->fe);
    ctx->n_faces = n_faces;
    ctx->nfn = nodes_per_face;
    std::vector<int32_t> fptr(N + 1, 0), finc, fsoa;
    std::vector<double> ft;
    if (n_faces > 0) {
        const int nfn = nodes_per_face;
        fsoa.resize((size_t)n_faces * nfn);
        for (int64_t f = 0; f < n_faces; ++f)
            for (int i = 0; i < nfn; ++i) {
                const int64_t v = face_conn[f * nfn + i] - index_base;
                if (v < 0 || v >= N) return jfm_fail(ctx, JFM_EINVAL, "face connectivity out of range");
                fsoa[(size_t)i * n_faces + f] = (int32_t)v;
                fptr[v + 1]++;
            }
        for (int64_t a = 0; a < N; ++a) fptr[a + 1] += fptr[a];
        finc.resize((size_t)n_faces * nfn);
        std::vector<int32_t> pos(fptr.begin(), fptr.end() - 1);
        for (int64_t f = 0; f < n_faces; ++f)
            for (int i = 0; i < nfn; ++i) finc[pos[fsoa[(size_t)i * n_faces + f]]++] = (int32_t)(f * nfn + i);
        ft.assign(traction, traction + 3 * n_faces);
        ALLOC(ctx, ctx->face_conn, int32_t, n_faces * nfn);
        ALLOC(ctx, ctx->face_t, double, 3 * n_faces);
        ALLOC(ctx, ctx->finc, int32_t, n_faces * nfn);
        ALLOC(ctx, ctx->fe, double, n_faces * nfn * 3);
        JFM_HIP(ctx, hipMemcpyAsync(ctx->face_conn, fsoa.data(), sizeof(int32_t) * fsoa.size(), hipMemcpyHostToDevice, s));
        JFM_HIP(ctx, hipMemcpyAsync(ctx->face_t, ft.data(), sizeof(double) * ft.size(), hipMemcpyHostToDevice, s));
        JFM_HIP(ctx, hipMemcpyAsync(ctx->finc, finc.data(), sizeof(int32_t) * finc.size(), hipMemcpyHostToDevice, s));
    }
    JFM_HIP(ctx, hipMemcpyAsync(ctx->finc_ptr, fptr.data(), sizeof(int32_t) * (N + 1), hipMemcpyHostToDevice, s));
    CHECK_LAUNCH(ctx, launch_face_loads(ctx));
    // the load of an unassembled problem is the external load
    JFM_HIP(ctx, hipMemcpyAsync(ctx->load, ctx->f_ext, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    if (int rc = sync(ctx)) return rc;
    ctx->has_bcs = true;
    ctx->has_load = true;
    jfem_learned_drop(ctx);
    ctx->learned_ready = false;
    ctx->has_user = false;
    for (Workspace *w : {&ctx->ws64, &ctx->ws32}) w->ok = false;  // preconditioners depend on the fixed set
    jfem_coarse_release(ctx);
    return JFM_OK;
}

// ================================================================ pattern ==
extern "C" int jfm_csr_pattern(jfm_ctx *ctx, int64_t *nnz_out, int64_t *rowptr, int64_t *colind, int32_t base) {
    if (!ctx) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (nnz_out) *nnz_out = 9 * ctx->nnzb;
    if (!rowptr && !colind) return JFM_OK;
    std::unique_lock<std::mutex> lock(ctx->pattern_mutex);
    if (ctx->h_brow.empty()) {  // the first call on this mesh
        JFM_HIP(ctx, hipSetDevice(ctx->device));
        std::vector<int32_t> br(ctx->N + 1);
        ctx->h_bcol.resize(ctx->nnzb);
        JFM_HIP(ctx, hipMemcpyAsync(br.data(), ctx->brow, 4 * br.size(), hipMemcpyDeviceToHost, ctx->stream));
        if (ctx->nnzb)
            JFM_HIP(ctx, hipMemcpyAsync(ctx->h_bcol.data(), ctx->bcol, 4 * ctx->h_bcol.size(), hipMemcpyDeviceToHost, ctx->stream));
        if (int rc = sync(ctx)) return rc;
        ctx->h_brow.swap(br);
    }
    lock.unlock();
    const std::vector<int32_t> &br = ctx->h_brow, &bc = ctx->h_bcol;
    parallel_for(ctx->N, 1024, [&](int64_t a0, int64_t a1) {
        for (int64_t a = a0; a < a1; ++a) {
            const int64_t r0 = br[a], nb = br[a + 1] - r0;
            for (int c = 0; c < 3; ++c) {
                const int64_t start = 9 * r0 + c * 3 * nb;
                if (rowptr) rowptr[3 * a + c] = start + base;
                if (colind)
                    for (int64_t k = 0; k < nb; ++k)
                        for (int d = 0; d < 3; ++d) colind[start + 3 * k + d] = 3 * (int64_t)bc[r0 + k] + d + base;
            }
        }
    });
    if (rowptr) rowptr[ctx->ndof] = 9 * ctx->nnzb + base;
    return JFM_OK;
}

// =============================================================== operator ==
template <typename T> static T *vals_of(jfm_ctx *ctx);
template <> double *vals_of<double>(jfm_ctx *ctx) { return ctx->vals64; }
template <> float *vals_of<float>(jfm_ctx *ctx) { return ctx->vals32; }

// the EBE operator's element matrices (FP64 and FP32, pair-major)
// With the patch operator, the element matrices are stored in its element
// order and the EBE product runs in the patch form (element results summed
// in LDS, shared nodes by the combine kernel).
static int ensure_element_matrices(jfm_ctx *ctx) {
    if (ctx->Ke) return JFM_OK;
    if (jfem_patch_enabled())
        if (int rc = jfem_patch_setup(ctx)) return rc;
    ALLOC(ctx, ctx->Ke, double, ctx->n_el * ke_stride(ctx->npair, 2));
    ALLOC(ctx, ctx->Ke32, float, ctx->n_el * ke_stride(ctx->npair, 4));
    ctx->ke_perm = ctx->patch_ready ? ctx->eperm : nullptr;
    CHECK_LAUNCH(ctx, launch_element_matrices(ctx));
    return JFM_OK;
}

// CSR values, each block recomputed from the geometric factors of its elements
static int ensure_assembled(jfm_ctx *ctx) {
    if (ctx->assembled) return JFM_OK;
    if (!ctx->vals64) ALLOC(ctx, ctx->vals64, double, 9 * ctx->nnzb);
    if (!ctx->vals32) ALLOC(ctx, ctx->vals32, float, 9 * ctx->nnzb);
    CHECK_LAUNCH(ctx, launch_assemble_values(ctx));
    ctx->assembled = true;
    return JFM_OK;
}

static int prepare_op(jfm_ctx *ctx, int op) {
    if (op == JFM_OP_CSR) return ensure_assembled(ctx);
    if (op == JFM_OP_EBE) return ensure_element_matrices(ctx);
    if (op == JFM_OP_MATFREE) return jfem_patch_enabled() ? jfem_patch_setup(ctx) : JFM_OK;
    if (op == kOpMass) return JFM_OK;
    if (op == kOpHeat) return ctx->heat_k ? JFM_OK : jfm_fail(ctx, JFM_ESTATE, "no heat problem uploaded");
    if (op == JFM_OP_TANGENT)
        return ctx->has_state ? JFM_OK
                              : jfm_fail(ctx, JFM_ESTATE, "tangent operator needs a state: call jfm_nl_residual first");
    return jfm_fail(ctx, JFM_EINVAL, "unknown operator variant");
}

// y = K x on free rows (fixed rows zeroed); optional partials of dot(y, dotv)
// into `part` (one per block of the last kernel, count in *npart).
template <typename T>
static hipError_t op_apply(jfm_ctx *ctx, int op, const T *x, T *y, const T *dotv, double *part, const int *done,
                           int *npart) {
    if (op == JFM_OP_CSR) return launch_bsr_spmv<T>(ctx, vals_of<T>(ctx), x, y, dotv, part, done, npart);
    if (op == kOpHeat) {
        if (sizeof(T) != 8) return hipErrorInvalidValue;
        return launch_heat_apply(ctx, (const double *)x, (double *)y, (const double *)dotv, part, done, npart);
    }
    return launch_two_phase<T>(ctx, op, x, y, dotv, part, done, npart);
}

// y = K x in FP64 outside of an iteration (residuals, reactions, internal
// forces).  The matrix-free product takes the patch form where the upload made the
// patches and not where an earlier call did: the two forms sum in different orders,
// and a mesh always gives the same bits.
static hipError_t op_product(jfm_ctx *ctx, int op, const double *x, double *y) {
    if (op != JFM_OP_MATFREE || ctx->patch_upload) return op_apply<double>(ctx, op, x, y, nullptr, nullptr, nullptr, nullptr);
    const hipError_t e = launch_elem_only<double>(ctx, op, x, nullptr);
    return e == hipSuccess ? launch_gather<double>(ctx, ctx->ye64, ctx->fixed, y, nullptr, nullptr, nullptr, nullptr) : e;
}

// Same without the row mask (all rows), for f_int and reactions.
static hipError_t op_product_all_rows(jfm_ctx *ctx, int op, const double *x, double *y) {
    uint8_t *saved = ctx->fixed;
    ctx->fixed = nullptr;
    hipError_t e = op_product(ctx, op, x, y);
    ctx->fixed = saved;
    return e;
}

extern "C" int jfm_apply(jfm_ctx *ctx, int32_t op, int32_t precision, const double *x, double *y) {
    if (!ctx || !x || !y) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (precision != JFM_FP64 && precision != JFM_FP32) return jfm_fail(ctx, JFM_EINVAL, "precision must be FP64 or FP32");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    if (int rc = prepare_op(ctx, op)) return rc;
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    JFM_HIP(ctx, hipMemcpyAsync(ctx->vx64, x, sizeof(double) * n, hipMemcpyHostToDevice, s));
    if (precision == JFM_FP64) {
        CHECK_LAUNCH(ctx, op_apply<double>(ctx, op, ctx->vx64, ctx->vy64, nullptr, nullptr, nullptr, nullptr));
    } else {
        CHECK_LAUNCH(ctx, (launch_convert<double, float>(ctx, ctx->vx64, ctx->vx32, n, 1.0)));
        CHECK_LAUNCH(ctx, op_apply<float>(ctx, op, ctx->vx32, ctx->vy32, nullptr, nullptr, nullptr, nullptr));
        CHECK_LAUNCH(ctx, (launch_convert<float, double>(ctx, ctx->vy32, ctx->vy64, n, 1.0)));
    }
    JFM_HIP(ctx, hipMemcpyAsync(y, ctx->vy64, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    return sync(ctx);
}

extern "C" int jfm_coarse_matrix(jfm_ctx *ctx, int32_t op, int32_t coarse_nodes, int64_t *nc, double *Ac,
                                 int32_t *node_agg) {
    if (!ctx || !nc || coarse_nodes <= 0) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (op != JFM_OP_MATFREE && op != JFM_OP_CSR && op != JFM_OP_TANGENT)
        return jfm_fail(ctx, JFM_EINVAL, "op must be MATFREE, CSR or TANGENT");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    return jfem_coarse_matrix(ctx, op, coarse_nodes, nc, Ac, node_agg);
}

extern "C" int jfm_time_apply(jfm_ctx *ctx, int32_t op, int32_t precision, int32_t reps, double *avg_ms) {
    if (!ctx || !avg_ms || reps <= 0) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (precision != JFM_FP64 && precision != JFM_FP32) return jfm_fail(ctx, JFM_EINVAL, "precision must be FP64 or FP32");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    if (int rc = prepare_op(ctx, op)) return rc;
    hipEvent_t t0, t1;
    JFM_HIP(ctx, hipEventCreate(&t0));
    JFM_HIP(ctx, hipEventCreate(&t1));
    const bool two = op != JFM_OP_CSR;
    const bool f64 = precision == JFM_FP64;
    // part 0: whole product, 1: SpMV or element phase, 2: gather
    auto run = [&](int part) -> hipError_t {
        if (!two) {
            return f64 ? launch_bsr_spmv<double>(ctx, ctx->vals64, ctx->vx64, ctx->vy64, nullptr, nullptr, nullptr, nullptr)
                       : launch_bsr_spmv<float>(ctx, ctx->vals32, ctx->vx32, ctx->vy32, nullptr, nullptr, nullptr, nullptr);
        }
        hipError_t e = hipSuccess;
        if (jfem_patch_form(ctx, op)) {  // patch kernel, then the shared-node kernel
            if (part != 2)
                e = f64 ? launch_patch_phase<double>(ctx, op, ctx->vx64, ctx->vy64, nullptr, nullptr)
                        : launch_patch_phase<float>(ctx, op, ctx->vx32, ctx->vy32, nullptr, nullptr);
            if (e != hipSuccess || part == 1) return e;
            return f64 ? launch_patch_combine<double>(ctx, ctx->vy64, nullptr, nullptr, nullptr, nullptr)
                       : launch_patch_combine<float>(ctx, ctx->vy32, nullptr, nullptr, nullptr, nullptr);
        }
        if (part != 2) e = f64 ? launch_elem_only<double>(ctx, op, ctx->vx64, nullptr) : launch_elem_only<float>(ctx, op, ctx->vx32, nullptr);
        if (e != hipSuccess || part == 1) return e;
        return f64 ? launch_gather<double>(ctx, ctx->ye64, ctx->fixed, ctx->vy64, nullptr, nullptr, nullptr, nullptr)
                   : launch_gather<float>(ctx, ctx->ye32, ctx->fixed, ctx->vy32, nullptr, nullptr, nullptr, nullptr);
    };
    // each part as `reps` back-to-back launches between two events, so the
    // averages are kernel durations plus launch gaps, without per-launch events
    for (int part = 0; part < (two ? 3 : 2); ++part) {
        CHECK_LAUNCH(ctx, run(part));  // warm
        JFM_HIP(ctx, hipEventRecord(t0, ctx->stream));
        for (int r = 0; r < reps; ++r) CHECK_LAUNCH(ctx, run(part));
        JFM_HIP(ctx, hipEventRecord(t1, ctx->stream));
        JFM_HIP(ctx, hipEventSynchronize(t1));
        float ms = 0.f;
        JFM_HIP(ctx, hipEventElapsedTime(&ms, t0, t1));
        avg_ms[part] = ms / reps;
    }
    if (!two) avg_ms[2] = 0.0;
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    return JFM_OK;
}

extern "C" int jfm_assemble(jfm_ctx *ctx, const double *u, double *vals, double *f) {
    if (!ctx) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    ctx->assembled = false;
    if (int rc = ensure_assembled(ctx)) return rc;
    const int64_t n = ctx->ndof;
    // f = f_ext - f_int(u)  (src/problems_elasticity.jl:432-433)
    if (u) {
        JFM_HIP(ctx, hipMemcpyAsync(ctx->vx64, u, sizeof(double) * n, hipMemcpyHostToDevice, s));
        CHECK_LAUNCH(ctx, op_product_all_rows(ctx, JFM_OP_MATFREE, ctx->vx64, ctx->vy64));
        CHECK_LAUNCH(ctx, (launch_convert<double, double>(ctx, ctx->vy64, ctx->vy64, n, -1.0)));
        std::vector<double> fi(n), fe(n);
        JFM_HIP(ctx, hipMemcpyAsync(fi.data(), ctx->vy64, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        JFM_HIP(ctx, hipMemcpyAsync(fe.data(), ctx->f_ext, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        if (int rc = sync(ctx)) return rc;
        for (int64_t i = 0; i < n; ++i) fe[i] += fi[i];
        JFM_HIP(ctx, hipMemcpyAsync(ctx->load, fe.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        if (int rc = sync(ctx)) return rc;
    } else {
        JFM_HIP(ctx, hipMemcpyAsync(ctx->load, ctx->f_ext, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    }
    ctx->has_load = true;
    if (vals) JFM_HIP(ctx, hipMemcpyAsync(vals, ctx->vals64, sizeof(double) * 9 * ctx->nnzb, hipMemcpyDeviceToHost, s));
    if (f) JFM_HIP(ctx, hipMemcpyAsync(f, ctx->load, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    return sync(ctx);
}

// Finite strain (finite_strain = true, src/problems_elasticity.jl:203-451):
// Km(u), Kg(u) and f = f_ext - f_int(u).  The device CSR operator then holds
// K = Km + Kg (Km alone without geometric stiffness), the K the reference
// solves (src/solvers.jl:286-292).
extern "C" int jfm_assemble_tl(jfm_ctx *ctx, int32_t geometric, const double *u, double *vals, double *vals_kg,
                               double *f) {
    if (!ctx) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (vals_kg && !geometric) return jfm_fail(ctx, JFM_EINVAL, "vals_kg requested without geometric stiffness");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    const int64_t n = ctx->ndof;
    const size_t vbytes = sizeof(double) * 9 * (size_t)ctx->nnzb;
    if (!ctx->vals64) ALLOC(ctx, ctx->vals64, double, 9 * ctx->nnzb);
    if (!ctx->vals32) ALLOC(ctx, ctx->vals32, float, 9 * ctx->nnzb);
    // finite-strain element blocks, the factors of Kg's, and the values of Km and
    // Kg that are asked for beside those of Km + Kg: a workspace that stays with the
    // mesh up to 512 MB (its allocation and release took 0.1 ms a call).  Where all
    // that does not fit, the element blocks alone, and Kg, Km and their sum one
    // after the other (three passes over elements and blocks instead of one).
    const int64_t pairs = ctx->n_el * ctx->npair, nv = 9 * ctx->nnzb, least = 9 * pairs;
    const int64_t want = least + (geometric ? pairs + (vals ? nv : 0) + (vals_kg ? nv : 0) : 0);
    bool one_pass = true;
    if (ctx->tl_ws_n < want) {
        free_ptr(ctx, ctx->tl_ws);
        ctx->tl_ws_n = 0;
        ctx->tl_ws = jfm_alloc<double>(ctx, want);
        one_pass = ctx->tl_ws != nullptr;
        if (!one_pass) ALLOC(ctx, ctx->tl_ws, double, least);
        ctx->tl_ws_n = one_pass ? want : least;
    }
    struct Keep {
        jfm_ctx *ctx;
        ~Keep() {
            if (ctx->tl_ws_n <= int64_t(64) << 20) return;
            (void)hipStreamSynchronize(ctx->stream);
            free_ptr(ctx, ctx->tl_ws);
            ctx->tl_ws_n = 0;
        }
    } keep{ctx};
    ctx->assembled = false;
    if (u) JFM_HIP(ctx, hipMemcpyAsync(ctx->vx64, u, sizeof(double) * n, hipMemcpyHostToDevice, s));
    else JFM_HIP(ctx, hipMemsetAsync(ctx->vx64, 0, sizeof(double) * n, s));
    // Km, Kg and the element forces; f = f_ext - f_int (src/problems_elasticity.jl:432-433)
    double *const ws = ctx->tl_ws;
    auto forces = [&]() -> int {
        CHECK_LAUNCH(ctx, launch_gather<double>(ctx, ctx->ye64, nullptr, ctx->vy64, nullptr, nullptr, nullptr, nullptr));
        CHECK_LAUNCH(ctx, (launch_convert<double, double>(ctx, ctx->vy64, ctx->vy64, n, -1.0)));
        CHECK_LAUNCH(ctx, launch_add(ctx, ctx->f_ext, ctx->vy64, ctx->load, n));
        return JFM_OK;
    };
    if (one_pass) {  // all launches before the copies, which the host waits in
        double *Kg = geometric ? ws + least : nullptr, *vm = geometric && vals ? Kg + pairs : nullptr;
        double *vg = geometric && vals_kg ? Kg + pairs + (vals ? nv : 0) : nullptr;
        CHECK_LAUNCH(ctx, launch_tl_element_matrices(ctx, ctx->vx64, ws, Kg, ctx->ye64));
        CHECK_LAUNCH(ctx, launch_assemble_values_ke(ctx, ws, Kg, vm, vg));
        if (int rc = forces()) return rc;
        if (vals_kg) JFM_HIP(ctx, hipMemcpyAsync(vals_kg, vg, vbytes, hipMemcpyDeviceToHost, s));
        if (vals) JFM_HIP(ctx, hipMemcpyAsync(vals, vm ? vm : ctx->vals64, vbytes, hipMemcpyDeviceToHost, s));
    } else {
        if (vals_kg) {
            CHECK_LAUNCH(ctx, launch_tl_element_matrices(ctx, ctx->vx64, nullptr, ws, nullptr));
            CHECK_LAUNCH(ctx, launch_assemble_values_kg(ctx, ws, false));
            JFM_HIP(ctx, hipMemcpyAsync(vals_kg, ctx->vals64, vbytes, hipMemcpyDeviceToHost, s));
        }
        CHECK_LAUNCH(ctx, launch_tl_element_matrices(ctx, ctx->vx64, ws, nullptr, ctx->ye64));
        CHECK_LAUNCH(ctx, launch_assemble_values_ke(ctx, ws, nullptr, nullptr, nullptr));
        if (int rc = forces()) return rc;
        if (vals) JFM_HIP(ctx, hipMemcpyAsync(vals, ctx->vals64, vbytes, hipMemcpyDeviceToHost, s));
        if (geometric) {
            CHECK_LAUNCH(ctx, launch_tl_element_matrices(ctx, ctx->vx64, nullptr, ws, nullptr));
            CHECK_LAUNCH(ctx, launch_assemble_values_kg(ctx, ws, true));
        }
    }
    if (f) JFM_HIP(ctx, hipMemcpyAsync(f, ctx->load, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    if (int rc = sync(ctx)) return rc;
    ctx->assembled = true;
    ctx->has_load = true;
    return JFM_OK;
}

// ================================================================ solvers ==
template <typename T> static Workspace &ws_of(jfm_ctx *ctx);
template <> Workspace &ws_of<double>(jfm_ctx *ctx) { return ctx->ws64; }
template <> Workspace &ws_of<float>(jfm_ctx *ctx) { return ctx->ws32; }

static int ensure_workspaces(jfm_ctx *ctx) {
    const int64_t n = ctx->ndof, N = ctx->N;
    if (!ctx->ws64.x) {
        Workspace &w = ctx->ws64;
        ALLOC(ctx, w.x, double, n); ALLOC(ctx, w.r, double, n); ALLOC(ctx, w.z, double, n);
        ALLOC(ctx, w.p, double, n); ALLOC(ctx, w.q, double, n); ALLOC(ctx, w.b, double, n);
        ALLOC(ctx, w.Minv, double, 9 * N);
    }
    if (!ctx->ws32.x) {
        Workspace &w = ctx->ws32;
        ALLOC(ctx, w.x, float, n); ALLOC(ctx, w.r, float, n); ALLOC(ctx, w.z, float, n);
        ALLOC(ctx, w.p, float, n); ALLOC(ctx, w.q, float, n); ALLOC(ctx, w.b, float, n);
        ALLOC(ctx, w.Minv, float, 9 * N);
    }
    if (!ctx->u64) ALLOC(ctx, ctx->u64, double, n);
    if (!ctx->rr64) ALLOC(ctx, ctx->rr64, double, n);
    if (!ctx->ws64.ok) {
        CHECK_LAUNCH(ctx, launch_block_jacobi(ctx, (double *)ctx->ws64.Minv, (float *)ctx->ws32.Minv));
        ctx->ws64.ok = ctx->ws32.ok = true;
    }
    return JFM_OK;
}

int jfem_ensure_workspaces(jfm_ctx *ctx) { return ensure_workspaces(ctx); }

static int read_scalars(jfm_ctx *ctx);
static int finalize_misc(jfm_ctx *ctx, int npart, int nv, int fin);

int jfem_dot(jfm_ctx *ctx, const double *a, const double *b, int64_t n, double *out) {
    int np = 0;
    CHECK_LAUNCH(ctx, launch_dot<double>(ctx, a, b, n, &np));
    if (int rc = finalize_misc(ctx, np, 1, FIN_DOT)) return rc;
    if (int rc = read_scalars(ctx)) return rc;
    *out = ctx->S_host->tmp0;
    return JFM_OK;
}

static int read_scalars(jfm_ctx *ctx) {
    JFM_HIP(ctx, hipMemcpyAsync(ctx->S_host, ctx->S, sizeof(PcgScalars), hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

// S_host is pinned and stream-ordered with the kernels that read S; the
// caller does not write S_host again before its next read_scalars, so no
// wait is needed here.
static int write_scalars(jfm_ctx *ctx) {
    JFM_HIP(ctx, hipMemcpyAsync(ctx->S, ctx->S_host, sizeof(PcgScalars), hipMemcpyHostToDevice, ctx->stream));
    return JFM_OK;
}

// One PCG iteration of parity `slot`: the operator, then the update and the
// direction (linalg_kernels.hip), with the coarse GEMV between them for the
// two-level preconditioner (coarse.hip); every kernel returns at once when
// done[slot] is set.
template <typename T>
static hipError_t pcg_iteration(jfm_ctx *ctx, int op, int slot, const T *Minv, bool coarse) {
    Workspace &w = ws_of<T>(ctx);
    T *x = (T *)w.x, *r = (T *)w.r, *z = (T *)w.z, *p = (T *)w.p, *q = (T *)w.q;
    int np_pq = 0, np_rz = 0;
    const bool fused = coarse && jfem_coarse_fused_restriction(ctx);
    // with the shared nodes' sums left to the update kernel, K p is the patch
    // kernel alone, its per-patch energies the p.q partials
    const bool defer = fused && jfem_patch_defer_shared(ctx, op);
    hipError_t e = defer ? launch_patch_phase<T>(ctx, op, p, q, p, &ctx->S->done[slot], ctx->partials + part_pq(slot))
                         : op_apply<T>(ctx, op, p, q, p, ctx->partials + part_pq(slot), &ctx->S->done[slot], &np_pq);
    if (e != hipSuccess) return e;
    if (defer) np_pq = ctx->npatch;
    if (fused) {
        // the update's blocks, one per aggregate, form w = Q' m r for the GEMV
        int np_wz = 0;
        e = launch_pcg_update<T>(ctx, slot, np_pq, x, r, z, p, q, Minv, &np_rz, nullptr, true, defer);
        if (e != hipSuccess) return e;
        e = launch_coarse_gemv_fused(ctx, slot, &np_wz);
        if (e != hipSuccess) return e;
        return launch_pcg_direction_coarse<T>(ctx, slot, np_rz, np_wz, p, z, x);  // x += alpha p here
    }
    // with the coarse level, the update also writes m o r in aggregate order
    T *rA = coarse ? coarse_rA<T>(ctx) : nullptr;
    e = launch_pcg_update<T>(ctx, slot, np_pq, x, r, z, p, q, Minv, &np_rz, rA);
    if (e != hipSuccess) return e;
    if (coarse) {  // zc = A_c^-1 Q' r, applied inside the direction update
        int np_wz = 0;
        e = launch_coarse_product_agg<T>(ctx, rA, &ctx->S->done[slot], &np_wz);
        if (e != hipSuccess) return e;
        return launch_pcg_direction_coarse<T>(ctx, slot, np_rz, np_wz, p, z, nullptr);
    }
    return launch_pcg_direction<T>(ctx, slot, np_rz, p, z);
}

bool jfem::jfem_use_graphs() {
    static const bool use = [] {
        const char *v = std::getenv("JFEM_GRAPHS");
        return !(v && v[0] == '0');
    }();
    return use;
}

// A batch of `batch` (even) iterations captured once as a HIP graph and
// replayed; kernels past convergence return immediately.
template <typename T>
static int pcg_batch(jfm_ctx *ctx, int op, const T *Minv, int batch, bool coarse) {
    const int prec = sizeof(T) == 8 ? JFM_FP64 : JFM_FP32;
    for (auto &g : ctx->graphs)
        if (g.op == op && g.prec == prec && g.minv == (const void *)Minv && g.batch == batch &&
            g.coarse == (coarse ? ctx->coarse_gen : 0)) {
            JFM_HIP(ctx, hipGraphLaunch(g.exec, ctx->stream));
            return JFM_OK;
        }
    if (!jfem_use_graphs()) {
        for (int it = 0; it < batch; ++it) CHECK_LAUNCH(ctx, pcg_iteration<T>(ctx, op, it & 1, Minv, coarse));
        return JFM_OK;
    }
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool ok = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal) == hipSuccess;
    hipError_t launch_err = hipSuccess;
    if (ok) {
        for (int it = 0; it < batch && launch_err == hipSuccess; ++it) launch_err = pcg_iteration<T>(ctx, op, it & 1, Minv, coarse);
        ok = hipStreamEndCapture(ctx->stream, &graph) == hipSuccess && launch_err == hipSuccess;
    }
    if (ok) ok = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess;
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    if (!ok) {  // capture unavailable: launch the same kernels directly
        if (exec) (void)hipGraphExecDestroy(exec);
        for (int it = 0; it < batch; ++it) CHECK_LAUNCH(ctx, pcg_iteration<T>(ctx, op, it & 1, Minv, coarse));
        return JFM_OK;
    }
    jfm_ctx::Graph g;
    g.op = op;
    g.prec = prec;
    g.minv = Minv;
    g.batch = batch;
    g.coarse = coarse ? ctx->coarse_gen : 0;
    g.exec = exec;
    ctx->graphs.push_back(g);
    JFM_HIP(ctx, hipGraphLaunch(exec, ctx->stream));
    return JFM_OK;
}

// sum of the misc partials -> scalars (one-block kernel)
static int finalize_misc(jfm_ctx *ctx, int npart, int nv, int fin) {
    CHECK_LAUNCH(ctx, launch_finalize(ctx, ctx->partials + kPartMisc, npart, nv, fin));
    return JFM_OK;
}

// The workgroups of resident kernels that run at once on a device, over all
// contexts and threads of the process, never exceed its CUs, each of which
// holds at least one of them: so every such kernel is resident as a whole once
// the finite kernels beside it have ended.  A kernel's workgroups go to the XCDs
// in turn and stay there, so a hold counts whole rounds of them: 85 workgroups are
// 11 on some XCD, and 85 + 85 + 86, 256 in all, would need 33 of its 32 CUs.  A hold
// lasts until the kernel has been waited for.
namespace {
struct ResidentHold {
    static constexpr int kDevices = 64;
    struct Device {
        std::mutex m;
        std::condition_variable cv;
        int used = 0;
    };
    static Device &of(int device) {
        static Device d[kDevices];
        return d[device % kDevices];
    }
    Device &dev;
    int n;
    ResidentHold(const jfm_ctx *ctx, int workgroups)
        : dev(of(ctx->device)), n(std::min((int)xcd_grid((unsigned)workgroups), ctx->cus)) {
        std::unique_lock<std::mutex> lock(dev.m);
        dev.cv.wait(lock, [&] { return dev.used + n <= ctx->cus; });
        dev.used += n;
    }
    ~ResidentHold() {
        {
            std::lock_guard<std::mutex> lock(dev.m);
            dev.used -= n;
        }
        dev.cv.notify_all();
    }
    ResidentHold(const ResidentHold &) = delete;
    ResidentHold &operator=(const ResidentHold &) = delete;
};
}  // namespace

// r = b - K x on the FP64 workspace, for a PCG that continues from x
static int warm_residual(jfm_ctx *ctx, int op) {
    const Workspace &w = ctx->ws64;
    int np = 0;
    CHECK_LAUNCH(ctx, op_product(ctx, op, (const double *)w.x, (double *)w.q));
    CHECK_LAUNCH(ctx, launch_residual(ctx, (const double *)w.b, (const double *)w.q, ctx->fixed, (double *)w.r, ctx->ndof, &np));
    return JFM_OK;
}

// PCG on the workspace of precision T: solves K x = b (free DOFs) from x = 0,
// or from the current x with its true residual (warm, FP64 only).  The host
// reads the scalars once per batch of `check_every` iterations.
template <typename T>
static int pcg_run(jfm_ctx *ctx, int op, const T *Minv, double rtol, int maxit, int check_every, int *iters,
                   int *status, bool warm = false, bool coarse = false) {
    Workspace &w = ws_of<T>(ctx);
    T *x = (T *)w.x, *r = (T *)w.r, *z = (T *)w.z, *p = (T *)w.p, *b = (T *)w.b;
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    const bool from_x = warm && sizeof(T) == 8;
    int np = 0;
    int resident = 1;
    if (int rc = jfem_persist_ready<T>(ctx, op, &resident, coarse)) return rc;
    if (resident) {
        if (from_x)
            if (int rc = warm_residual(ctx, op)) return rc;
        const ResidentHold hold(ctx, jfem_persist_workgroups(ctx, op));  // until the kernel has ended
        T *out = from_x ? z : x;
        CHECK_LAUNCH(ctx, launch_pcg_persist<T>(ctx, op, Minv, b, from_x ? x : nullptr, from_x ? r : nullptr, out, rtol, maxit, coarse));
        if (int rc = read_scalars(ctx)) return rc;
        if (!ctx->S_host->fail) {
            if (from_x) JFM_HIP(ctx, hipMemcpyAsync(x, out, sizeof(T) * n, hipMemcpyDeviceToDevice, s));
            ++ctx->resident_solves;
            ctx->persist_fails = 0;
            *iters = ctx->S_host->iter;
            *status = ctx->S_host->done[0];
            return JFM_OK;
        }
        resident_gave_up(ctx, 1);  // launched below
    }
    if (int rc = prepare_op(ctx, op)) return rc;
    std::memset(ctx->S_host, 0, sizeof(PcgScalars));
    ctx->S_host->rtol2 = rtol * rtol;
    ctx->S_host->maxit = maxit;
    if (int rc = write_scalars(ctx)) return rc;
    if (from_x) {
        // restart from the current x with the true residual r = b - K x
        if (int rc = warm_residual(ctx, op)) return rc;
    } else {
        JFM_HIP(ctx, hipMemsetAsync(x, 0, sizeof(T) * n, s));
        JFM_HIP(ctx, hipMemcpyAsync(r, b, sizeof(T) * n, hipMemcpyDeviceToDevice, s));
    }
    CHECK_LAUNCH(ctx, launch_dot<T>(ctx, b, b, n, &np));
    if (int rc = finalize_misc(ctx, np, 1, FIN_BB)) return rc;
    const bool ordered = coarse && jfem_coarse_fused_restriction(ctx);
    if (ordered)
        if (int rc = jfem_coarse_order(ctx)) return rc;
    CHECK_LAUNCH(ctx, launch_pcg_init<T>(ctx, r, z, p, Minv, &np, ordered));
    if (coarse) CHECK_LAUNCH(ctx, launch_coarse_correct<T>(ctx, r, z, p, ctx->partials + kPartMisc, nullptr, &np));
    if (ordered) {
        if (int rc = jfem_patch_qsrc(ctx)) return rc;
        Minv = (const T *)ctx->MA;  // what the iterations read (one captured graph for all blocks)
    }
    if (int rc = finalize_misc(ctx, np, 2, FIN_INIT)) return rc;
    // Batches of up to check_every iterations; once the residual falls, the
    // next batch is the power of two that covers the iterations its rate
    // predicts are left, so that few launches run past convergence.  The
    // first batch follows the start without a host read (its kernels return
    // at once if the start already converged); the start's r.r comes back
    // with the first batch's scalars (rr0).
    const int bmax = std::max(2, (check_every + 1) & ~1);
    int batch = bmax;
    double rr_prev = -1.0;
    int it_prev = 0;
    for (bool first = true; first || ctx->S_host->done[0] == DONE_RUNNING; first = false) {
        if (int rc = pcg_batch<T>(ctx, op, Minv, batch, coarse)) return rc;
        if (int rc = read_scalars(ctx)) return rc;
        if (first) rr_prev = ctx->S_host->rr0;
        const double rr = ctx->S_host->rr, tol2 = ctx->S_host->tol2;
        const int it = ctx->S_host->iter;
        batch = bmax;
        if (rr > tol2 && tol2 > 0.0 && rr < rr_prev && it > it_prev) {
            const double left = std::log(tol2 / rr) / (std::log(rr / rr_prev) / (it - it_prev));
            int nb = 2;
            while (nb < left + 1.0 && nb < bmax) nb *= 2;
            batch = std::min(nb, bmax);
        }
        rr_prev = rr;
        it_prev = it;
    }
    *iters = ctx->S_host->iter;
    *status = ctx->S_host->done[0];
    return JFM_OK;
}

// FP64 true residual r = b - K u over free DOFs; *rnorm = |r|.
static int true_residual(jfm_ctx *ctx, int op, const double *b, const double *u, double *r, double *rnorm) {
    int np = 0;
    CHECK_LAUNCH(ctx, op_product(ctx, op, u, ctx->vy64));
    CHECK_LAUNCH(ctx, launch_residual(ctx, b, ctx->vy64, ctx->fixed, r, ctx->ndof, &np));
    if (int rc = finalize_misc(ctx, np, 1, FIN_DOT)) return rc;
    if (int rc = read_scalars(ctx)) return rc;
    *rnorm = std::sqrt(ctx->S_host->tmp0);
    return JFM_OK;
}

// Learned blocks against block Jacobi for the system in ws64.b: builds the
// learned blocks from the block Jacobi now in ws*.Minv, then, with probe > 0,
// runs `probe` PCG iterations from 0 with each.  After the same number of
// iterations the iterate with the larger energy b.x_k (CG decreases
// 1/2 x'Kx - b.x = -1/2 b.x_k monotonically) has the smaller energy-norm
// error; the learned blocks are kept only if they win.
static int learned_select(jfm_ctx *ctx, int op, int probe, int check, bool *use, int *iters, double *setup_ms,
                          bool coarse) {
    double lms = 0.0;
    if (int rc = jfem_learned_prepare(ctx, setup_ms ? &lms : nullptr)) return rc;
    if (setup_ms) *setup_ms += lms;
    *use = true;
    if (probe <= 0) return JFM_OK;
    // The probe runs in FP32 (FP32 operator and blocks) on b rounded to FP32:
    // it only ranks the two preconditioners by the energy b'x_k.
    double phi[2] = {0.0, 0.0};
    const float *cand[2] = {(const float *)ctx->ws32.Minv, ctx->Mlearn32};
    const int64_t n = ctx->ndof;
    if (!ctx->xprobe) ALLOC(ctx, ctx->xprobe, double, n);
    double *xd[2] = {ctx->xprobe, ctx->vy64};  // the iterates in FP64 (vy64 is free here)
    CHECK_LAUNCH(ctx, (launch_convert<double, float>(ctx, (const double *)ctx->ws64.b, (float *)ctx->ws32.b, n, 1.0)));
    for (int c = 0; c < 2; ++c) {
        int it = 0, status = 0;
        if (int rc = pcg_run<float>(ctx, op, cand[c], 1e-30, probe, check, &it, &status, false, coarse)) return rc;
        CHECK_LAUNCH(ctx, (launch_convert<float, double>(ctx, (const float *)ctx->ws32.x, xd[c], n, 1.0)));
        if (int rc = jfem_dot(ctx, (const double *)ctx->ws64.b, xd[c], n, &phi[c])) return rc;
        *iters += it;
    }
    *use = phi[1] > phi[0];
    // the winner's probe iterate starts the solve
    if (*use) JFM_HIP(ctx, hipMemcpyAsync(ctx->xprobe, xd[1], sizeof(double) * n, hipMemcpyDeviceToDevice, ctx->stream));
    return JFM_OK;
}

extern "C" int jfm_solve(jfm_ctx *ctx, const jfm_solve_opts *opts, const double *f, double *u, double *la,
                         jfm_solve_stats *stats) {
    if (!ctx || !opts || !u) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (!f && !ctx->has_load) return jfm_fail(ctx, JFM_ESTATE, "no load vector: upload BCs or pass f");
    if (!(opts->rtol > 0.0) || opts->maxit <= 0) return jfm_fail(ctx, JFM_EINVAL, "rtol > 0 and maxit > 0 required");
    if (opts->method != JFM_SOLVE_PCG && opts->method != JFM_SOLVE_MIXED_IR)
        return jfm_fail(ctx, JFM_EINVAL, "unknown solve method");
    if (opts->precond != JFM_PREC_BLOCK_JACOBI && opts->precond != JFM_PREC_LEARNED && opts->precond != JFM_PREC_USER)
        return jfm_fail(ctx, JFM_EINVAL, "unknown preconditioner");
    if (opts->precond == JFM_PREC_USER && !ctx->has_user)
        return jfm_fail(ctx, JFM_ESTATE, "no user preconditioner blocks set");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    resident_begin(ctx);
    const int op = opts->op;
    const int op_outer = opts->method == JFM_SOLVE_MIXED_IR ? opts->op_outer : op;
    // The 480-element patches of the matrix-free operator serve launched
    // iterations (and, made with the upload, op_product): where the iterations may
    // run resident, pcg_run makes them if it has to launch after all.
    const bool inner32 = opts->method == JFM_SOLVE_MIXED_IR;
    const bool resident = inner32 ? jfem_persist_maybe<float>(ctx, op) : jfem_persist_maybe<double>(ctx, op);
    if (op != JFM_OP_MATFREE || !resident)
        if (int rc = prepare_op(ctx, op)) return rc;
    if (op_outer != JFM_OP_MATFREE)
        if (int rc = prepare_op(ctx, op_outer)) return rc;
    if (int rc = ensure_workspaces(ctx)) return rc;
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    const int check = std::max(2, opts->check_every > 0 ? opts->check_every : 32);
    jfm_solve_stats st{};
    hipEvent_t e0, e1;
    JFM_HIP(ctx, hipEventCreate(&e0));
    JFM_HIP(ctx, hipEventCreate(&e1));

    // right-hand side b = f - K g on free rows (elimination of prescribed
    // DOFs, src/solvers.jl:206-210); f stays in vx64 for the reactions
    if (f) JFM_HIP(ctx, hipMemcpyAsync(ctx->vx64, f, sizeof(double) * n, hipMemcpyHostToDevice, s));
    else JFM_HIP(ctx, hipMemcpyAsync(ctx->vx64, ctx->load, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    double *b = (double *)ctx->ws64.b;
    JFM_HIP(ctx, hipEventRecord(e0, s));
    double bnorm = 0.0;
    if (int rc = true_residual(ctx, op_outer, ctx->vx64, ctx->g, b, &bnorm)) return rc;
    ctx->hist_it.clear();
    ctx->hist_res.clear();
    const bool coarse = opts->coarse_nodes > 0 && bnorm > 0.0;
    // the learned blocks on a second stream beside the coarse level's
    // inversion (both read only the mesh and the block Jacobi)
    if (coarse)
        if (int rc = jfem_coarse_setup(ctx, op_outer, opts->coarse_nodes, &st.setup_ms,
                                       opts->precond == JFM_PREC_LEARNED)) {
            jfem_learned_drop(ctx);  // no learned work is left running past the call
            return rc;
        }
    const double *Minv64 = (const double *)ctx->ws64.Minv;
    const float *Minv32 = (const float *)ctx->ws32.Minv;
    if (opts->precond == JFM_PREC_USER) {
        Minv64 = ctx->Muser64;
        Minv32 = ctx->Muser32;
    }
    const double *x0 = nullptr;  // initial iterate (b = f - K g system), when a probe made one
    if (opts->precond == JFM_PREC_LEARNED && bnorm > 0.0) {
        bool use = true;
        int its = 0;
        if (int rc = learned_select(ctx, op_outer, opts->learned_probe, check, &use, &its, &st.setup_ms, coarse))
            return rc;
        st.iterations += its;
        x0 = opts->learned_probe > 0 ? ctx->xprobe : nullptr;
        if (use) {
            Minv64 = ctx->Mlearn64;
            Minv32 = ctx->Mlearn32;
        } else {
            st.fallback = 1;
        }
    }

    if (bnorm == 0.0) {
        JFM_HIP(ctx, hipMemcpyAsync(ctx->u64, ctx->g, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    } else if (opts->method == JFM_SOLVE_PCG) {
        int it = 0, status = 0, total = 0, restarts = 0;
        if (x0) JFM_HIP(ctx, hipMemcpyAsync(ctx->ws64.x, x0, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        if (int rc = pcg_run<double>(ctx, op, Minv64, opts->rtol, opts->maxit, check, &it, &status, x0 != nullptr,
                                     coarse))
            return rc;
        total = it;
        // The recursive residual drifts from the true one near the FP64 floor:
        // restart from x with the true residual until it meets rtol (residual
        // replacement), a bounded number of times.
        while (status == DONE_CONVERGED && restarts < 8 && total < opts->maxit) {
            double rn = 0.0;
            if (int rc = true_residual(ctx, op, b, (const double *)ctx->ws64.x, ctx->rr64, &rn)) return rc;
            ctx->hist_it.push_back(total);
            ctx->hist_res.push_back(rn / bnorm);
            if (rn <= opts->rtol * bnorm) break;
            if (int rc = pcg_run<double>(ctx, op, Minv64, opts->rtol, opts->maxit - total, check, &it, &status, true,
                                         coarse))
                return rc;
            total += it;
            ++restarts;
        }
        st.iterations += total;
        st.outer = 1 + restarts;
        // u = x + g
        CHECK_LAUNCH(ctx, launch_add(ctx, ctx->g, (const double *)ctx->ws64.x, ctx->u64, n));
    } else {
        // FP64 iterative refinement around FP32 PCG: r = f - K u in FP64,
        // K d = r / |r| in FP32 to inner_rtol, u += |r| d.
        if (x0) CHECK_LAUNCH(ctx, launch_add(ctx, ctx->g, x0, ctx->u64, n));
        else JFM_HIP(ctx, hipMemcpyAsync(ctx->u64, ctx->g, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        int total = 0, outer = 0;
        const double inner = opts->inner_rtol > 0 ? opts->inner_rtol : 1e-4;
        const int max_outer = opts->max_outer > 0 ? opts->max_outer : 20;
        if (opts->first_rtol > 0.0) {
            // FP64 phase for the smooth low modes that FP32 cannot resolve
            int it = 0, status = 0;
            if (x0) JFM_HIP(ctx, hipMemcpyAsync(ctx->ws64.x, x0, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
            if (int rc = pcg_run<double>(ctx, op_outer, Minv64, opts->first_rtol, opts->maxit, check, &it, &status,
                                         x0 != nullptr, coarse))
                return rc;
            total += it;
            CHECK_LAUNCH(ctx, launch_add(ctx, ctx->g, (const double *)ctx->ws64.x, ctx->u64, n));
        }
        while (outer < max_outer) {
            double rn = 0.0;
            if (int rc = true_residual(ctx, op_outer, ctx->vx64, ctx->u64, ctx->rr64, &rn)) return rc;
            ctx->hist_it.push_back(total);
            ctx->hist_res.push_back(rn / bnorm);
            if (rn <= opts->rtol * bnorm || total >= opts->maxit) break;
            CHECK_LAUNCH(ctx, (launch_convert<double, float>(ctx, ctx->rr64, (float *)ctx->ws32.b, n, 1.0 / rn)));
            int it = 0, status = 0;
            int cap = opts->maxit - total;
            if (opts->inner_maxit > 0) cap = std::min(cap, opts->inner_maxit);
            // spread the remaining reduction (to 0.3 x the target) evenly over
            // the fewest inner solves that each reduce by at most inner_rtol:
            // the last solve then ends well below the target instead of just
            // above it, and no solve asks FP32 for more than inner_rtol
            double rt = inner;
            const double R = 0.3 * opts->rtol * bnorm / rn;
            if (R < 1.0 && inner < 1.0) {
                const int k = std::max(1, (int)std::ceil(std::log(R) / std::log(inner) - 1e-9));
                rt = std::pow(R, 1.0 / k);
            }
            if (int rc = pcg_run<float>(ctx, op, Minv32, rt, cap, check, &it, &status, false, coarse)) return rc;
            total += it;
            ++outer;
            CHECK_LAUNCH(ctx, launch_axpy_scaled(ctx, ctx->u64, (const float *)ctx->ws32.x, rn, n));
            if (status == DONE_BREAKDOWN) break;
        }
        st.iterations += total;
        st.outer = outer;
    }
    // final FP64 true residual with the FP64 operator
    double rn = 0.0;
    if (int rc = true_residual(ctx, op_outer, ctx->vx64, ctx->u64, ctx->rr64, &rn)) return rc;
    JFM_HIP(ctx, hipEventRecord(e1, s));
    JFM_HIP(ctx, hipEventSynchronize(e1));
    float ms = 0.f;
    JFM_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    st.relres = bnorm > 0 ? rn / bnorm : 0.0;
    st.converged = st.relres <= opts->rtol ? 1 : 0;
    st.solve_ms = ms;
    JFM_HIP(ctx, hipMemcpyAsync(u, ctx->u64, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    if (la) {
        // la = f - K u on fixed DOFs (src/solvers.jl:212-213), 0 elsewhere
        CHECK_LAUNCH(ctx, op_product_all_rows(ctx, op_outer, ctx->u64, ctx->vy64));
        std::vector<double> ku(n), ff(n);
        std::vector<uint8_t> fxd(n);
        JFM_HIP(ctx, hipMemcpyAsync(ku.data(), ctx->vy64, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        JFM_HIP(ctx, hipMemcpyAsync(ff.data(), ctx->vx64, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        JFM_HIP(ctx, hipMemcpyAsync(fxd.data(), ctx->fixed, n, hipMemcpyDeviceToHost, s));
        if (int rc = sync(ctx)) return rc;
        for (int64_t i = 0; i < n; ++i) la[i] = fxd[i] ? ff[i] - ku[i] : 0.0;
    }
    if (int rc = sync(ctx)) return rc;
    if (stats) *stats = st;
    if (!st.converged) {
        char msg[160];
        std::snprintf(msg, sizeof msg, "solver did not reach rtol %.3e: relres %.3e after %d iterations", opts->rtol,
                      st.relres, st.iterations);
        return jfm_fail(ctx, JFM_ENOCONV, msg);
    }
    return JFM_OK;
}

extern "C" int jfm_solve_history(jfm_ctx *ctx, int32_t *iterations, double *relres, int32_t max_entries) {
    if (!ctx || max_entries < 0) return JFM_EINVAL;
    const int n = std::min<int>(max_entries, (int)ctx->hist_it.size());
    for (int k = 0; k < n; ++k) {
        if (iterations) iterations[k] = ctx->hist_it[k];
        if (relres) relres[k] = ctx->hist_res[k];
    }
    return n;
}

extern "C" int jfm_precond_set_blocks(jfm_ctx *ctx, const double *M) {
    if (!ctx || !M) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    const int64_t N = ctx->N;
    std::vector<double> m(M, M + 9 * N);
    std::vector<uint8_t> fx(3 * N);
    JFM_HIP(ctx, hipMemcpyAsync(fx.data(), ctx->fixed, 3 * N, hipMemcpyDeviceToHost, ctx->stream));
    if (int rc = sync(ctx)) return rc;
    std::vector<float> m32(9 * N);
    for (int64_t a = 0; a < N; ++a)
        for (int c = 0; c < 3; ++c) {
            for (int d = 0; d < 3; ++d) {
                if (fx[3 * a + c] || fx[3 * a + d]) m[9 * a + 3 * c + d] = 0.0;
                if (!std::isfinite(m[9 * a + 3 * c + d])) return jfm_fail(ctx, JFM_EINVAL, "non-finite preconditioner block");
            }
        }
    for (int64_t k = 0; k < 9 * N; ++k) m32[k] = (float)m[k];
    if (!ctx->Muser64) ALLOC(ctx, ctx->Muser64, double, 9 * N);
    if (!ctx->Muser32) ALLOC(ctx, ctx->Muser32, float, 9 * N);
    JFM_HIP(ctx, hipMemcpyAsync(ctx->Muser64, m.data(), sizeof(double) * 9 * N, hipMemcpyHostToDevice, ctx->stream));
    JFM_HIP(ctx, hipMemcpyAsync(ctx->Muser32, m32.data(), sizeof(float) * 9 * N, hipMemcpyHostToDevice, ctx->stream));
    if (int rc = sync(ctx)) return rc;
    ctx->has_user = true;
    return JFM_OK;
}

// ============================================================== nonlinear ==
static int nl_buffers(jfm_ctx *ctx) {
    const int64_t n = ctx->ndof, N = ctx->N;
    if (!ctx->ustate64) ALLOC(ctx, ctx->ustate64, double, n);
    if (!ctx->ustate32) ALLOC(ctx, ctx->ustate32, float, n);
    if (!ctx->Dtan) ALLOC(ctx, ctx->Dtan, double, 9 * N);
    if (!ctx->nl_u) ALLOC(ctx, ctx->nl_u, double, n);
    if (!ctx->nl_r) ALLOC(ctx, ctx->nl_r, double, n);
    if (!ctx->nl_du) ALLOC(ctx, ctx->nl_du, double, n);
    if (!ctx->nl_zero) {
        ALLOC(ctx, ctx->nl_zero, double, n);
        JFM_HIP(ctx, hipMemsetAsync(ctx->nl_zero, 0, sizeof(double) * n, ctx->stream));
    }
    return JFM_OK;
}

// Makes u (device, n_dofs) the state of the tangent operator and computes
// R = lf f_ext - f_int(u) on the free DOFs (0 on fixed ones), *rnorm = |R|
// (NAN when some Gauss point has det F <= 0).  Uses vx64/vy64 as scratch.
static int nl_residual(jfm_ctx *ctx, const double *u, double lf, double *R, double *rnorm) {
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    if (u != ctx->ustate64) JFM_HIP(ctx, hipMemcpyAsync(ctx->ustate64, u, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    CHECK_LAUNCH(ctx, (launch_convert<double, float>(ctx, ctx->ustate64, ctx->ustate32, n, 1.0)));
    ctx->has_state = true;
    int np = 0;
    CHECK_LAUNCH(ctx, launch_nh_elem<double>(ctx, false, ctx->gf64, ctx->ustate64, nullptr, ctx->ye64, nullptr));
    CHECK_LAUNCH(ctx, launch_gather<double>(ctx, ctx->ye64, ctx->fixed, ctx->vy64, nullptr, nullptr, nullptr, &np));
    CHECK_LAUNCH(ctx, (launch_convert<double, double>(ctx, ctx->f_ext, ctx->vx64, n, lf)));
    CHECK_LAUNCH(ctx, launch_residual(ctx, ctx->vx64, ctx->vy64, ctx->fixed, R, n, &np));
    if (int rc = finalize_misc(ctx, np, 1, FIN_DOT)) return rc;
    if (int rc = read_scalars(ctx)) return rc;
    *rnorm = std::sqrt(ctx->S_host->tmp0);
    return JFM_OK;
}

extern "C" int jfm_nl_residual(jfm_ctx *ctx, const double *u, double load_factor, double *R, double *rnorm) {
    if (!ctx || !u) return JFM_EINVAL;
    if (!ctx->has_mesh || !ctx->has_bcs) return jfm_fail(ctx, JFM_ESTATE, "upload the mesh and boundary conditions first");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    if (int rc = nl_buffers(ctx)) return rc;
    const int64_t n = ctx->ndof;
    JFM_HIP(ctx, hipMemcpyAsync(ctx->nl_u, u, sizeof(double) * n, hipMemcpyHostToDevice, ctx->stream));
    double rn = 0.0;
    if (int rc = nl_residual(ctx, ctx->nl_u, load_factor, ctx->nl_r, &rn)) return rc;
    if (R) JFM_HIP(ctx, hipMemcpyAsync(R, ctx->nl_r, sizeof(double) * n, hipMemcpyDeviceToHost, ctx->stream));
    if (int rc = sync(ctx)) return rc;
    if (rnorm) *rnorm = rn;
    return JFM_OK;
}

// K_T du = r (r in nl_r, free DOFs) to |r - K_T du| <= eta |r|; du -> nl_du.
static int tangent_solve(jfm_ctx *ctx, const jfm_newton_opts *o, const double *M64, const float *M32, double eta,
                         double rnorm, int check, bool coarse, int *iters) {
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    *iters = 0;
    if (o->method == JFM_SOLVE_PCG) {
        JFM_HIP(ctx, hipMemcpyAsync(ctx->ws64.b, ctx->nl_r, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        int it = 0, status = 0;
        if (int rc = pcg_run<double>(ctx, JFM_OP_TANGENT, M64, eta, o->maxit_linear, check, &it, &status, false,
                                     coarse))
            return rc;
        *iters = it;
        JFM_HIP(ctx, hipMemcpyAsync(ctx->nl_du, ctx->ws64.x, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        return JFM_OK;
    }
    // FP32 PCG inside FP64 refinement on the tangent
    JFM_HIP(ctx, hipMemsetAsync(ctx->nl_du, 0, sizeof(double) * n, s));
    const double inner = o->inner_rtol > 0 ? o->inner_rtol : 1e-2;
    double rl = rnorm;
    for (int outer = 0; outer < 50; ++outer) {
        if (outer > 0)
            if (int rc = true_residual(ctx, JFM_OP_TANGENT, ctx->nl_r, ctx->nl_du, ctx->rr64, &rl)) return rc;
        if (rl <= eta * rnorm || *iters >= o->maxit_linear) break;
        const double *src = outer == 0 ? ctx->nl_r : ctx->rr64;
        CHECK_LAUNCH(ctx, (launch_convert<double, float>(ctx, src, (float *)ctx->ws32.b, n, 1.0 / rl)));
        int it = 0, status = 0;
        int cap = o->maxit_linear - *iters;
        if (o->inner_maxit > 0) cap = std::min(cap, o->inner_maxit);
        // no need to solve the correction beyond what the outer tolerance asks
        const double tol = std::max(inner, 0.5 * eta * rnorm / rl);
        if (int rc = pcg_run<float>(ctx, JFM_OP_TANGENT, M32, tol, cap, check, &it, &status, false, coarse)) return rc;
        *iters += it;
        CHECK_LAUNCH(ctx, launch_axpy_scaled(ctx, ctx->nl_du, (const float *)ctx->ws32.x, rl, n));
        if (status == DONE_BREAKDOWN) break;
    }
    return JFM_OK;
}

extern "C" int jfm_solve_nonlinear(jfm_ctx *ctx, const jfm_newton_opts *opts, double *u, jfm_newton_stats *stats) {
    if (!ctx || !opts || !u) return JFM_EINVAL;
    if (!ctx->has_mesh || !ctx->has_bcs) return jfm_fail(ctx, JFM_ESTATE, "upload the mesh and boundary conditions first");
    if (opts->load_steps < 1 || opts->max_newton < 1 || !(opts->rtol > 0.0) || opts->maxit_linear < 1)
        return jfm_fail(ctx, JFM_EINVAL, "load_steps, max_newton, maxit_linear >= 1 and rtol > 0 required");
    if (opts->method != JFM_SOLVE_PCG && opts->method != JFM_SOLVE_MIXED_IR)
        return jfm_fail(ctx, JFM_EINVAL, "unknown solve method");
    if (opts->precond != JFM_PREC_BLOCK_JACOBI && opts->precond != JFM_PREC_LEARNED)
        return jfm_fail(ctx, JFM_EINVAL, "the tangent solves take JFM_PREC_BLOCK_JACOBI or JFM_PREC_LEARNED");
    if (opts->precond == JFM_PREC_LEARNED && !ctx->has_mlp)
        return jfm_fail(ctx, JFM_ESTATE, "learned preconditioner requested but no weights are loaded");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    resident_begin(ctx);
    if (int rc = ensure_workspaces(ctx)) return rc;
    if (int rc = nl_buffers(ctx)) return rc;
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    const int check = std::max(2, opts->check_every > 0 ? opts->check_every : 32);
    const double eta_max = opts->eta_max > 0.0 && opts->eta_max < 1.0 ? opts->eta_max : 0.1;
    static const bool verbose = [] {
        const char *v = std::getenv("JFEM_VERBOSE");
        return v && v[0] == '1';
    }();
    jfm_newton_stats st{};
    ctx->hist_it.clear();
    ctx->hist_res.clear();
    hipEvent_t e0, e1;
    JFM_HIP(ctx, hipEventCreate(&e0));
    JFM_HIP(ctx, hipEventCreate(&e1));
    JFM_HIP(ctx, hipEventRecord(e0, s));
    // |f_ext| on the free DOFs
    double fnorm = 0.0;
    {
        int np = 0;
        CHECK_LAUNCH(ctx, launch_residual(ctx, ctx->f_ext, ctx->nl_zero, ctx->fixed, ctx->rr64, n, &np));
        if (int rc = finalize_misc(ctx, np, 1, FIN_DOT)) return rc;
        if (int rc = read_scalars(ctx)) return rc;
        fnorm = std::sqrt(ctx->S_host->tmp0);
    }
    JFM_HIP(ctx, hipMemsetAsync(ctx->nl_u, 0, sizeof(double) * n, s));
    bool all_ok = true;
    double relres = 0.0;
    struct Restore {  // the workspaces end with the tangent block Jacobi: rebuild the linear one on next use
        jfm_ctx *c;
        ~Restore() {
            c->ws64.ok = c->ws32.ok = false;
            c->minv_tangent = false;
            jfem_learned_drop(c);
            c->learned_ready = false;
        }
    } restore{ctx};
    for (int step = 1; step <= opts->load_steps && all_ok; ++step) {
        const double lf = (double)step / opts->load_steps, lf0 = (double)(step - 1) / opts->load_steps;
        // prescribed displacements follow the load factor (g is zero on free DOFs)
        if (ctx->g_nonzero) {
            CHECK_LAUNCH(ctx, (launch_convert<double, double>(ctx, ctx->g, ctx->rr64, n, lf - lf0)));
            CHECK_LAUNCH(ctx, launch_add(ctx, ctx->nl_u, ctx->rr64, ctx->nl_u, n));
        }
        double rn = 0.0;
        if (int rc = nl_residual(ctx, ctx->nl_u, lf, ctx->nl_r, &rn)) return rc;
        if (!std::isfinite(rn))
            return jfm_fail(ctx, JFM_ENOCONV, "inadmissible state (det F <= 0) at the start of a load step");
        const double ref = lf * fnorm > 0.0 ? lf * fnorm : (rn > 0.0 ? rn : 1.0);
        bool ok = false;
        double rn_prev = rn, eta_prev = eta_max;
        bool step_learned = true;  // this load step's probe outcome
        for (int it = 0;; ++it) {
            relres = rn / ref;
            ctx->hist_it.push_back(st.linear_iterations);
            ctx->hist_res.push_back(relres);
            if (rn <= opts->rtol * ref) { ok = true; break; }
            if (it >= opts->max_newton) break;
            // tangent block Jacobi at the current state (features use its diagonal)
            CHECK_LAUNCH(ctx, launch_nh_block_jacobi(ctx, ctx->ustate64, (double *)ctx->ws64.Minv, (float *)ctx->ws32.Minv,
                                                     ctx->Dtan));
            ctx->ws64.ok = ctx->ws32.ok = true;
            ctx->minv_tangent = true;
            const bool coarse = opts->coarse_nodes > 0;
            // coarse level of the tangent, rebuilt at the first iterate of each
            // load step; later iterates keep it (Q A_c^-1 Q' stays SPD, only
            // less exact as K_T moves)
            if (coarse && it == 0)
                if (int rc = jfem_coarse_setup(ctx, JFM_OP_TANGENT, opts->coarse_nodes, nullptr)) return rc;
            const double *M64 = (const double *)ctx->ws64.Minv;
            const float *M32 = (const float *)ctx->ws32.Minv;
            if (opts->precond == JFM_PREC_LEARNED) {
                // The probe runs at the first iterate of each load step, like the
                // coarse rebuild; later iterates of the step keep its outcome.
                // Accepted blocks are recomputed from the new tangent diagonal at
                // every Newton step.
                jfem_learned_drop(ctx);
                ctx->learned_ready = false;
                bool use = false;
                int its = 0;
                if (it == 0 || step_learned) {
                    JFM_HIP(ctx, hipMemcpyAsync(ctx->ws64.b, ctx->nl_r, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
                    const int probe = it == 0 ? opts->learned_probe : 0;
                    if (int rc = learned_select(ctx, JFM_OP_TANGENT, probe, check, &use, &its, nullptr, coarse))
                        return rc;
                    if (it == 0) step_learned = use;
                }
                st.linear_iterations += its;
                if (use) {
                    M64 = ctx->Mlearn64;
                    M32 = ctx->Mlearn32;
                } else {
                    ++st.fallbacks;
                }
            }
            // Forcing term.  The reference uses min(0.9, |R|^0.5) on the absolute
            // residual (ext/JuliaFEMCUDAExt.jl:785-787), which is unit dependent
            // and near 0.9 for a relative one; here Eisenstat-Walker choice 2,
            // eta = 0.9 (|R_k| / |R_k-1|)^2 with their safeguard, starting each
            // load step at eta_max, capped by eta_max and never tighter than the
            // Newton tolerance needs.
            double eta = eta_max;
            if (it > 0) {
                const double ratio = rn / rn_prev;
                eta = 0.9 * ratio * ratio;
                const double safe = 0.9 * eta_prev * eta_prev;
                if (safe > 0.1) eta = std::max(eta, safe);
                eta = std::min(eta, eta_max);
            }
            eta = std::max(eta, 0.5 * opts->rtol * ref / rn);
            eta_prev = eta;
            rn_prev = rn;
            int lits = 0;
            if (int rc = tangent_solve(ctx, opts, M64, M32, eta, rn, check, coarse, &lits)) return rc;
            st.linear_iterations += lits;
            ++st.newton_iterations;
            if (verbose)
                std::fprintf(stderr, "[jfem] load step %d/%d, Newton %d: relres %.3e, eta %.2e, %d PCG iterations\n",
                             step, opts->load_steps, it + 1, relres, eta, lits);
            // u += du; halve the step while some Gauss point leaves det F > 0
            JFM_HIP(ctx, hipMemcpyAsync(ctx->rr64, ctx->nl_u, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
            double rnew = 0.0;
            for (int bt = 0;; ++bt) {
                CHECK_LAUNCH(ctx, launch_add(ctx, ctx->rr64, ctx->nl_du, ctx->nl_u, n));
                if (int rc = nl_residual(ctx, ctx->nl_u, lf, ctx->nl_r, &rnew)) return rc;
                if (std::isfinite(rnew) || bt >= 12) break;
                CHECK_LAUNCH(ctx, (launch_convert<double, double>(ctx, ctx->nl_du, ctx->nl_du, n, 0.5)));
            }
            if (!std::isfinite(rnew)) break;
            rn = rnew;
        }
        all_ok = ok;
    }
    JFM_HIP(ctx, hipEventRecord(e1, s));
    JFM_HIP(ctx, hipEventSynchronize(e1));
    float ms = 0.f;
    JFM_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    JFM_HIP(ctx, hipMemcpyAsync(u, ctx->nl_u, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    if (int rc = sync(ctx)) return rc;
    st.converged = all_ok ? 1 : 0;
    st.relres = relres;
    st.solve_ms = ms;
    if (stats) *stats = st;
    if (!all_ok) {
        char msg[160];
        std::snprintf(msg, sizeof msg, "Newton did not reach rtol %.3e: relres %.3e after %d iterations", opts->rtol,
                      relres, st.newton_iterations);
        return jfm_fail(ctx, JFM_ENOCONV, msg);
    }
    return JFM_OK;
}

// ========================================================= postprocessing ==
// M x_k = b_k for the nsys right-hand sides at b + k n, x likewise, beside of them
// side by side in the resident PCG (M the consistent mass, Mm its inverse diagonal);
// *done: false after a give-up.
static int mass_solves(jfm_ctx *ctx, const double *Mm, int nsys, int beside, const double *b, double *x, bool *done) {
    const int64_t n = ctx->ndof;
    hipStream_t s = ctx->stream;
    std::vector<PcgScalars> S(beside);  // (outlives the copy into it)
    *done = false;
    for (int k = 0; k < nsys; k += beside) {
        const ResidentHold hold(ctx, beside * ctx->cells.npatch);
        CHECK_LAUNCH(ctx, launch_pcg_persist<double>(ctx, kOpMass, Mm, b + k * n, nullptr, nullptr, x + k * n, 1e-13, 2000, false, beside, n));
        JFM_HIP(ctx, hipMemcpyAsync(S.data(), ctx->cells.S, sizeof(PcgScalars) * beside, hipMemcpyDeviceToHost, s));
        if (int rc = sync(ctx)) return rc;
        int failed = 0;
        for (const PcgScalars &v : S) failed += v.fail != 0;
        ctx->resident_solves += beside - failed;
        if (failed) {
            resident_gave_up(ctx, failed);
            return JFM_OK;
        }
    }
    ctx->persist_fails = 0;
    *done = true;
    return JFM_OK;
}

extern "C" int jfm_postprocess(jfm_ctx *ctx, const double *u, double *strain_gp, double *stress_gp,
                               double *strain_nodal, double *stress_nodal) {
    if (!ctx || !u) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    resident_begin(ctx);
    if (int rc = ensure_workspaces(ctx)) return rc;
    const int64_t n = ctx->ndof, N = ctx->N, nq = ctx->n_el * ctx->ngp * 6;
    hipStream_t s = ctx->stream;
    // the fits are one operator with two right-hand sides per field, all of them
    // side by side where the resident PCG takes them; their vectors are in one
    // allocation with the diagonal (three of their own cost 0.4 ms a call, of 11
    // at 65,000 Hex8)
    double *outs[2] = {strain_nodal, stress_nodal};
    int nf = 0, field[2];
    for (int f = 0; f < 2; ++f)
        if (outs[f]) field[nf++] = f;
    const int nsys = 2 * nf;
    int beside = nsys;
    if (nsys)
        if (int rc = jfem_persist_ready<double>(ctx, kOpMass, &beside)) return rc;
    const int64_t kept = beside > 1 ? nsys : std::min(nsys, 1);  // solutions
    double *du = jfm_alloc<double>(ctx, n), *eps = jfm_alloc<double>(ctx, nq), *sig = jfm_alloc<double>(ctx, nq),
           *Mm = jfm_alloc<double>(ctx, 9 * N + (nsys ? kept * n + 6 * N : 0) + (beside > 1 ? nsys * n : 0));
    auto cleanup = [&] {
        for (void *p : {(void *)du, (void *)eps, (void *)sig, (void *)Mm}) jfm_free(ctx, p);
    };
    if (!du || !eps || !sig || !Mm) {
        cleanup();
        return jfm_fail(ctx, JFM_ENOMEM, "device allocation failed in jfm_postprocess");
    }
    int rc = JFM_OK;
    auto fail_hip = [&](hipError_t e, const char *what) {
        rc = jfm_hip_fail(ctx, e, what);
        return rc;
    };
    hipError_t e = hipMemcpyAsync(du, u, sizeof(double) * n, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = launch_post_gp(ctx, du, eps, sig);
    if (e != hipSuccess) fail_hip(e, "launch_post_gp");
    if (rc == JFM_OK && strain_gp) {
        e = hipMemcpyAsync(strain_gp, eps, sizeof(double) * nq, hipMemcpyDeviceToHost, s);
        if (e != hipSuccess) fail_hip(e, "strain copy");
    }
    if (rc == JFM_OK && stress_gp) {
        e = hipMemcpyAsync(stress_gp, sig, sizeof(double) * nq, hipMemcpyDeviceToHost, s);
        if (e != hipSuccess) fail_hip(e, "stress copy");
    }
    // nodal least-squares fits (src/problems_elasticity.jl:550-594): M x = b
    // per three components, PCG with the mass operator and its diagonal
    if (rc == JFM_OK && nsys) {
        e = launch_mass_diag(ctx, Mm);
        if (e != hipSuccess) fail_hip(e, "launch_mass_diag");
        double *J = Mm + 9 * N, *X = J + 6 * N, *B = X + kept * n;
        bool done = false;
        if (beside > 1) {
            for (int k = 0; k < nsys && rc == JFM_OK; ++k)
                if ((e = launch_post_rhs(ctx, du, field[k / 2], 3 * (k % 2), B + k * n)) != hipSuccess) fail_hip(e, "launch_post_rhs");
            if (rc == JFM_OK) rc = mass_solves(ctx, Mm, nsys, beside, B, X, &done);
        }
        for (int f = 0; f < nf && rc == JFM_OK; ++f) {
            const double *x0 = X, *x1 = (const double *)ctx->ws64.x;
            if (done) {
                x0 = X + 2 * f * n;
                x1 = x0 + n;
            }
            for (int h = 0; h < 2 && !done && rc == JFM_OK; ++h) {
                int it = 0, status = 0;
                if ((e = launch_post_rhs(ctx, du, field[f], 3 * h, (double *)ctx->ws64.b)) != hipSuccess) fail_hip(e, "launch_post_rhs");
                if (rc == JFM_OK) rc = pcg_run<double>(ctx, kOpMass, Mm, 1e-13, 2000, 32, &it, &status);
                if (rc == JFM_OK && h == 0) {
                    e = hipMemcpyAsync(X, ctx->ws64.x, sizeof(double) * n, hipMemcpyDeviceToDevice, s);
                    if (e != hipSuccess) fail_hip(e, "nodal copy");
                }
            }
            if (rc != JFM_OK) break;
            e = launch_post_join(ctx, x0, x1, J);
            if (e == hipSuccess) e = hipMemcpyAsync(outs[field[f]], J, sizeof(double) * 6 * N, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) fail_hip(e, "nodal copy");
        }
    }
    e = hipStreamSynchronize(s);
    if (rc == JFM_OK && e != hipSuccess) fail_hip(e, "jfm_postprocess");
    cleanup();
    return rc;
}

// ================================================================== heat ==
extern "C" int jfm_heat_solve(jfm_ctx *ctx, const double *k, const double *q, int64_t n_faces, int32_t nodes_per_face,
                              const int64_t *face_conn, const double *flux, const double *h, const double *T_ext,
                              const uint8_t *fixed_node, const double *T_fixed, int32_t index_base, double rtol,
                              int32_t maxit, double *T, jfm_solve_stats *stats) {
    if (!ctx || !k || !T || !(rtol > 0.0) || maxit <= 0) return JFM_EINVAL;
    if (!ctx->has_mesh) return jfm_fail(ctx, JFM_ESTATE, "no mesh");
    if (n_faces < 0 || (n_faces > 0 && !face_conn)) return jfm_fail(ctx, JFM_EINVAL, "invalid face arguments");
    if (n_faces > 0 && nodes_per_face != 6 && nodes_per_face != 3 && nodes_per_face != 4)
        return jfm_fail(ctx, JFM_EUNSUPPORTED, "nodes_per_face must be 6 (Tri6), 3 (Tri3) or 4 (Quad4)");
    if ((h == nullptr) != (T_ext == nullptr)) return jfm_fail(ctx, JFM_EINVAL, "convection needs both h and T_ext");
    JFM_HIP(ctx, hipSetDevice(ctx->device));
    resident_begin(ctx);
    if (int rc = ensure_workspaces(ctx)) return rc;
    const int64_t N = ctx->N, n = ctx->ndof, n_el = ctx->n_el;
    hipStream_t s = ctx->stream;
    for (int64_t e = 0; e < n_el; ++e)
        if (!(k[e] > 0.0)) return jfm_fail(ctx, JFM_EINVAL, "thermal conductivity must be positive");
    // the captured PCG graphs of a previous heat problem point at its buffers
    drop_graphs(ctx);
    release_heat(ctx);
    ALLOC(ctx, ctx->heat_k, double, n_el);
    ALLOC(ctx, ctx->heat_fixed, uint8_t, n);
    ALLOC(ctx, ctx->heat_g, double, n);
    ALLOC(ctx, ctx->heat_Minv, double, 9 * N);
    JFM_HIP(ctx, hipMemcpyAsync(ctx->heat_k, k, sizeof(double) * n_el, hipMemcpyHostToDevice, s));
    std::vector<uint8_t> fx(n, 1);
    std::vector<double> g(n, 0.0);
    for (int64_t a = 0; a < N; ++a) {
        fx[3 * a] = fixed_node ? fixed_node[a] : 0;
        if (fx[3 * a] && T_fixed) g[3 * a] = T_fixed[a];
    }
    JFM_HIP(ctx, hipMemcpyAsync(ctx->heat_fixed, fx.data(), n, hipMemcpyHostToDevice, s));
    JFM_HIP(ctx, hipMemcpyAsync(ctx->heat_g, g.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
    double *src = nullptr;
    if (q) {
        src = jfm_alloc<double>(ctx, n_el);
        if (!src) return jfm_fail(ctx, JFM_ENOMEM, "device allocation failed in jfm_heat_solve");
        JFM_HIP(ctx, hipMemcpyAsync(src, q, sizeof(double) * n_el, hipMemcpyHostToDevice, s));
    }
    if (n_faces > 0) {
        const int nfn = nodes_per_face;
        std::vector<int32_t> soa((size_t)n_faces * nfn), fptr(N + 1, 0);
        for (int64_t f = 0; f < n_faces; ++f)
            for (int i = 0; i < nfn; ++i) {
                const int64_t v = face_conn[f * nfn + i] - index_base;
                if (v < 0 || v >= N) {
                    if (src) jfm_free(ctx, src);
                    return jfm_fail(ctx, JFM_EINVAL, "face connectivity out of range");
                }
                soa[(size_t)i * n_faces + f] = (int32_t)v;
                fptr[v + 1]++;
            }
        for (int64_t a = 0; a < N; ++a) fptr[a + 1] += fptr[a];
        std::vector<int32_t> inc((size_t)n_faces * nfn), pos(fptr.begin(), fptr.end() - 1);
        for (int64_t f = 0; f < n_faces; ++f)  // ascending face order per node
            for (int i = 0; i < nfn; ++i) inc[pos[soa[(size_t)i * n_faces + f]]++] = (int32_t)(f * nfn + i);
        ctx->hf_n = n_faces;
        ctx->hf_nfn = nfn;
        ALLOC(ctx, ctx->hf_conn, int32_t, n_faces * nfn);
        ALLOC(ctx, ctx->hf_ptr, int32_t, N + 1);
        ALLOC(ctx, ctx->hf_inc, int32_t, n_faces * nfn);
        ALLOC(ctx, ctx->hf_fe, double, n_faces * nfn * 3);
        JFM_HIP(ctx, hipMemcpyAsync(ctx->hf_conn, soa.data(), 4 * soa.size(), hipMemcpyHostToDevice, s));
        JFM_HIP(ctx, hipMemcpyAsync(ctx->hf_ptr, fptr.data(), 4 * (N + 1), hipMemcpyHostToDevice, s));
        JFM_HIP(ctx, hipMemcpyAsync(ctx->hf_inc, inc.data(), 4 * inc.size(), hipMemcpyHostToDevice, s));
        for (auto [dst, v] : {std::pair<double **, const double *>{&ctx->hf_g, flux}, {&ctx->hf_h, h}, {&ctx->hf_text, T_ext}})
            if (v) {
                ALLOC(ctx, *dst, double, n_faces);
                JFM_HIP(ctx, hipMemcpyAsync(*dst, v, sizeof(double) * n_faces, hipMemcpyHostToDevice, s));
            }
    }
    if (int rc = jfem_heat_faces(ctx)) return rc;
    // the heat row mask stands in for the elasticity one for this solve
    struct MaskSwap {
        jfm_ctx *c;
        uint8_t *saved;
        ~MaskSwap() { c->fixed = saved; }
    } swap{ctx, ctx->fixed};
    ctx->fixed = ctx->heat_fixed;
    hipEvent_t e0, e1;
    JFM_HIP(ctx, hipEventCreate(&e0));
    JFM_HIP(ctx, hipEventCreate(&e1));
    JFM_HIP(ctx, hipEventRecord(e0, s));
    jfm_solve_stats st{};
    // b = f - K g on the free temperatures
    CHECK_LAUNCH(ctx, launch_heat_load(ctx, src, ctx->vx64));
    double *b = (double *)ctx->ws64.b;
    double bnorm = 0.0;
    if (int rc = true_residual(ctx, kOpHeat, ctx->vx64, ctx->heat_g, b, &bnorm)) return rc;
    CHECK_LAUNCH(ctx, launch_heat_jacobi(ctx, ctx->heat_Minv));
    const int check = 32;
    if (bnorm > 0.0) {
        int it = 0, status = 0, total = 0;
        if (int rc = pcg_run<double>(ctx, kOpHeat, ctx->heat_Minv, rtol, maxit, check, &it, &status)) return rc;
        total = it;
        for (int restart = 0; restart < 4 && total < maxit; ++restart) {  // residual replacement, as jfm_solve
            double rn = 0.0;
            if (int rc = true_residual(ctx, kOpHeat, b, (const double *)ctx->ws64.x, ctx->rr64, &rn)) return rc;
            if (rn <= rtol * bnorm) break;
            if (int rc = pcg_run<double>(ctx, kOpHeat, ctx->heat_Minv, rtol, maxit - total, check, &it, &status, true))
                return rc;
            total += it;
            st.outer++;
        }
        st.iterations = total;
        CHECK_LAUNCH(ctx, launch_add(ctx, ctx->heat_g, (const double *)ctx->ws64.x, ctx->u64, n));
    } else {
        JFM_HIP(ctx, hipMemcpyAsync(ctx->u64, ctx->heat_g, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    }
    double rn = 0.0;
    if (int rc = true_residual(ctx, kOpHeat, ctx->vx64, ctx->u64, ctx->rr64, &rn)) return rc;
    JFM_HIP(ctx, hipEventRecord(e1, s));
    JFM_HIP(ctx, hipEventSynchronize(e1));
    float ms = 0.f;
    JFM_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    std::vector<double> u(n);
    JFM_HIP(ctx, hipMemcpyAsync(u.data(), ctx->u64, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    if (int rc = sync(ctx)) return rc;
    if (src) jfm_free(ctx, src);
    for (int64_t a = 0; a < N; ++a) T[a] = u[3 * a];
    st.relres = bnorm > 0.0 ? rn / bnorm : 0.0;
    st.converged = st.relres <= rtol ? 1 : 0;
    st.solve_ms = ms;
    if (stats) *stats = st;
    if (!st.converged) return jfm_fail(ctx, JFM_ENOCONV, "heat solve did not reach rtol");
    return JFM_OK;
}
