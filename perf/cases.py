"""Timed cases: what a user of the library runs, through its public entry points.

listed() gives the cases, draw() more of the same ranges, prepare() what a
program holds before the call, run() one pass, work() its unavoidable bytes
and operations, exact() the same results from plain torch in 64 bits.

Kinds (`case["kind"]`):
  ku        K.u on device vectors (a caller's own iteration, jfm_apply_noalloc)
  solve     one linear solve of an uploaded problem (Context.solve)
  new_mesh  a whole linear analysis of a mesh seen for the first time: upload,
            boundary conditions, solve
  nonlinear load-stepped neo-Hookean Newton (Context.solve_nonlinear)
  heat      steady conduction with source, flux and convection
  post      stresses and strains at Gauss points and nodes
  assemble  CSR values and load vector handed to the host
  tl        finite-strain assembly (Km, Kg, f) handed to the host, the matrix
            of each iteration of a host-driven Newton loop
  train     one gradient of the learned preconditioner (forward + backward)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "juliafem.jl_amd"))

import jfem  # noqa: E402
from jfem import mesh as M  # noqa: E402
from jfem.learned import DEFAULT_WEIGHTS  # noqa: E402

F64 = torch.float64
GEN = {"Tet10": M.box_tet10, "Tet4": M.box_tet4, "Hex8": M.box_hex8}
NPE = {"Tet10": 10, "Tet4": 4, "Hex8": 8}
NGP = {"Tet10": 4, "Tet4": 1, "Hex8": 8}

# solver settings in use: the library's default call, the assembled operator,
# the two-level forms of the benchmark (FP64, FP32 inside FP64 refinement, and
# the same with the learned blocks probed)
METHODS = {
    "pcg": dict(),
    "pcg_csr": dict(op="csr", op_outer="csr"),
    "two_level": dict(check_every=16),
    "mixed": dict(method=1, inner_rtol=2e-3, check_every=16),
    "learned": dict(method=1, precond=1, learned_probe=16, inner_rtol=2e-3, check_every=16),
}


def _coarse(nx, ny, nz):
    """Nodes per aggregate: the benchmark's 1,536 at its size, fewer on small meshes."""
    return 1536 if nx * ny * nz >= 20000 else 256


def listed():
    def c(name, kind, etype, grid, **kw):
        return dict(name=name, kind=kind, etype=etype, nx=grid[0], ny=grid[1], nz=grid[2], **kw)

    return [
        # the smallest analysis in use (the smoke test's cantilever): launches and latency
        c("solve_smallest", "solve", "Tet10", (10, 2, 2), method="pcg", rtol=1e-10),
        # default solve() call on an ordinary mesh (139,587 DOFs)
        c("solve_default", "solve", "Tet10", (80, 8, 8), method="pcg", rtol=1e-8),
        # assembled operator and reactions, hexahedra, odd sizes
        c("solve_csr_hex", "solve", "Hex8", (41, 5, 7), method="pcg_csr", rtol=1e-9),
        # the benchmark's headline: 1,048,707 DOFs, learned blocks probed, FP32 in FP64 refinement
        c("solve_headline", "solve", "Tet10", (160, 16, 16), method="learned", rtol=1e-8),
        # one analysis of a new mesh, odd sizes
        c("new_mesh", "new_mesh", "Tet10", (61, 7, 5), method="mixed", rtol=1e-8),
        # K.u for a caller's own iteration at 1,048,707 DOFs
        c("ku_large", "ku", "Tet10", (160, 16, 16)),
        # finite deformation, two load steps
        c("nonlinear", "nonlinear", "Tet10", (60, 6, 6), steps=2),
        # conduction with convection on the end face
        c("heat", "heat", "Tet10", (80, 8, 8)),
        # recovery of stresses and strains after a solve
        c("postprocess", "post", "Tet10", (60, 6, 6)),
        # K and f to the host (a host direct solver, or the reference's own)
        c("assemble", "assemble", "Tet10", (60, 6, 6)),
        # finite-strain K of a host-driven Newton iteration, odd sizes
        c("assemble_tl", "tl", "Tet10", (37, 3, 5)),
        # a training step of the learned preconditioner, four residual/error pairs
        c("train_grad", "train", "Tet10", (60, 6, 6), pairs=4),
    ]


# the largest number of hexes along x drawn per kind, and for the solves without a
# coarse level (thousands of iterations), so that no drawn case costs more than the listed ones
TOP = {"ku": 160, "solve": 110, "new_mesh": 64, "nonlinear": 60, "heat": 100, "post": 80, "assemble": 70, "tl": 40, "train": 80}
TOP_ONE_LEVEL = 60


def draw(rng):
    kind = rng.choice(list(TOP))
    lo, hi = 8, TOP[kind]
    etype = "Tet10" if kind == "train" else rng.choice(["Tet10", "Tet10", "Tet10", "Hex8", "Tet4"])
    case = dict(kind=kind, etype=etype)
    if kind in ("solve", "new_mesh"):
        case["method"] = rng.choice(["pcg", "pcg_csr", "two_level", "mixed", "learned"] if kind == "solve" else ["pcg", "two_level", "mixed"])
        if case["method"] in ("pcg", "pcg_csr"):
            hi = TOP_ONE_LEVEL
    nx = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    ny, nz = (max(2, int(round(nx / 10 * rng.uniform(0.6, 1.3)))) for _ in range(2))
    case.update(nx=nx, ny=ny, nz=nz)
    if "method" in case:
        case["rtol"] = 1e-10 if nx < 24 else (1e-9 if nx < 50 else 1e-8)
    if kind == "nonlinear":
        case["steps"] = rng.randint(1, 3)
    if kind == "train":
        case["pairs"] = rng.randint(2, 6)
    return case


# ------------------------------------------------------------------ inputs ---
def _mesh(case, seed):
    nl = case["kind"] == "nonlinear"
    r = np.random.default_rng(seed)
    # a cantilever of fixed length, its hexes near cubes, jittered, log-normal stiffness;
    # the nonlinear one deflects by about 10% of its span
    t = -52.5 * r.uniform(0.7, 1.0) if nl else -r.uniform(0.5, 1.5)
    sec = (10.0 * case["ny"] / case["nx"], 10.0 * case["nz"] / case["nx"])
    if nl:
        t *= min(sec) ** 2  # bending stiffness of the section
    return GEN[case["etype"]](case["nx"], case["ny"], case["nz"], L=(10.0,) + sec, seed=int(seed), jitter=0.1,
                              E_sigma=0.3 if nl else 0.5, traction=(0.0, 0.0, t))


def _displacement(m, seed, size):
    """A smooth bending field with some roughness, zero on the clamp."""
    r = np.random.default_rng(seed + 1)
    x = m.X[:, 0] / 10.0
    u = np.stack([0.1 * x * np.sin(2.0 * m.X[:, 1]), 0.3 * x ** 2, -x ** 2 * (1.5 - 0.5 * x)], axis=1) * r.uniform(0.5, 1.0)
    u = size * (u + 0.002 * r.standard_normal(u.shape))
    u[m.clamp_nodes] = 0.0
    return np.ascontiguousarray(u.reshape(-1))


def _heat_inputs(m, seed):
    r = np.random.default_rng(seed + 2)
    nf = m.faces.shape[0]
    return dict(k=np.exp(0.5 * r.standard_normal(m.n_el)) * 3.0, q=r.uniform(0.5, 2.0, m.n_el), faces=m.faces,
                flux=r.uniform(0.0, 1.0, nf), h=r.uniform(0.5, 1.0, nf), T_ext=r.uniform(10.0, 20.0, nf),
                fixed=np.isclose(m.X[:, 0], 0.0).astype(np.uint8), T_fixed=np.full(m.n_nodes, 5.0))


def _pairs(m, seed, n):
    """Residual / error pairs (r = K e): errors of a half-converged iteration are smooth with a rough part."""
    K = _Elements(m).stiffness()
    E, R = [], []
    for p in range(n):
        e = _displacement(m, seed + 10 + p, 1e-4 * (1 + p))
        E.append(e)
        y = K.times(torch.from_numpy(e).to(K.dev))
        y[torch.from_numpy(m.fixed_mask().astype(bool)).to(K.dev)] = 0.0
        R.append(y.cpu().numpy())
    return np.array(R), np.array(E)


def prepare(case, seed):
    m = _mesh(case, seed)
    kind = case["kind"]
    s = dict(case=case, ctx=jfem.Context(0), mesh=m)
    ctx = s["ctx"]
    if kind == "new_mesh":
        s["fixed"], s["traction"] = m.fixed_mask(), m.face_traction()
        return s
    ctx.upload(m)
    if kind == "ku":
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        s["x"] = torch.randn(m.n_dofs, dtype=F64, device="cuda", generator=g)
        s["y"] = torch.empty_like(s["x"])
    elif kind == "solve" and case["method"] == "learned":
        with open(DEFAULT_WEIGHTS, "rb") as fh:
            s["weights"] = fh.read()
        ctx.set_learned_weights(s["weights"])
    elif kind == "heat":
        s["heat"] = _heat_inputs(m, seed)
    elif kind in ("post", "assemble"):
        s["u"] = _displacement(m, seed, 1e-3)
    elif kind == "tl":
        s["u"] = _displacement(m, seed, 0.5)
    elif kind == "train":
        s["R"], s["E"] = _pairs(m, seed, case["pairs"])
        with open(DEFAULT_WEIGHTS, "rb") as fh:
            s["weights"] = fh.read()
    return s


def _solve_kw(case):
    kw = dict(rtol=case["rtol"], **METHODS[case["method"]])
    if case["method"] in ("two_level", "mixed", "learned"):
        kw["coarse_nodes"] = _coarse(case["nx"], case["ny"], case["nz"])
    return kw


def run(state):
    ctx, m, case = state["ctx"], state["mesh"], state["case"]
    kind = case["kind"]
    if kind == "ku":
        rc = ctx._lib.jfm_apply_noalloc(ctx._h, 2, 0, ctypes.c_void_p(state["x"].data_ptr()), ctypes.c_void_p(state["y"].data_ptr()),
                                        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(f"jfm_apply_noalloc: {rc}")
        return state["y"]
    if kind == "solve":
        if "weights" in state:  # as in a training or evaluation loop: the blocks follow the weights
            ctx.set_learned_weights(state["weights"])
        u, la, _ = ctx.solve(want_la=case["method"] == "pcg_csr", **_solve_kw(case))
        return u if la is None else (u, la)
    if kind == "new_mesh":
        ctx.upload_mesh(m.X, m.conn, m.etype, m.E, m.nu)
        ctx.upload_bcs(state["fixed"], None, m.faces, m.ftype, state["traction"])
        return ctx.solve(**_solve_kw(case))[0]
    if kind == "nonlinear":
        return ctx.solve_nonlinear(load_steps=case["steps"], rtol=1e-8, method=1, inner_rtol=1e-2,
                                   coarse_nodes=_coarse(case["nx"], case["ny"], case["nz"]))[0]
    if kind == "heat":
        return ctx.heat_solve(**state["heat"])[0]
    if kind == "post":
        return ctx.postprocess(state["u"])
    if kind == "assemble":
        return ctx.assemble(state["u"])
    if kind == "tl":
        return ctx.assemble_tl(state["u"])
    ctx.set_learned_weights(state["weights"])
    return ctx.learned_grad(state["R"], state["E"])


def _sizes(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["etype"] == "Tet10":
        return (2 * nx + 1) * (2 * ny + 1) * (2 * nz + 1), 6 * nx * ny * nz
    return (nx + 1) * (ny + 1) * (nz + 1), (6 if case["etype"] == "Tet4" else 1) * nx * ny * nz


def work(case):
    """Inputs read once and outputs written once (a solve's iterations are the method's own)."""
    N, n_el = _sizes(case)
    npe, ngp = NPE[case["etype"]], NGP[case["etype"]]
    mesh = 24 * N + 4 * npe * n_el + 16 * n_el
    per_k = n_el * ngp * npe * (12 + 6 * 3)        # one K.u, gradients and nodal forces
    adj = {"Tet10": 27.7, "Tet4": 14.5, "Hex8": 26.0}[case["etype"]]
    kind = case["kind"]
    if kind == "ku":
        return {"bytes": mesh + 48 * N, "flops": per_k}
    if kind in ("solve", "new_mesh", "nonlinear"):
        return {"bytes": mesh + 48 * N, "flops": per_k * (1 if kind != "nonlinear" else 4 * case["steps"])}
    if kind == "heat":
        return {"bytes": mesh + 16 * N + 16 * n_el, "flops": per_k // 3}
    if kind == "post":
        return {"bytes": mesh + 24 * N + 96 * ngp * n_el + 96 * N, "flops": per_k}
    blocks = n_el * ngp * npe * (npe + 1) // 2 * 30
    if kind == "assemble":
        return {"bytes": mesh + 24 * N + 24 * N + 72 * adj * N, "flops": per_k + blocks}
    if kind == "tl":
        return {"bytes": mesh + 24 * N + 24 * N + 144 * adj * N, "flops": per_k + 2 * blocks}
    return {"bytes": mesh + 48 * N * case["pairs"] + 4 * 6150, "flops": per_k * case["pairs"] + 3 * 12032 * N}


# ------------------------------------------------- 64-bit values, plain torch ---
def _basis(etype, p):
    """(N, dN/dxi) of the element at reference points p (n, 3), from the shape functions' definitions."""
    x, y, z = p[:, 0], p[:, 1], p[:, 2]
    if etype == "Hex8":
        c = np.array([(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1)], float)
        f = 1 + c[None] * p[:, None]
        Nv = f.prod(2) / 8
        d = np.stack([c[:, k] * f[:, :, (k + 1) % 3] * f[:, :, (k + 2) % 3] / 8 for k in range(3)], axis=2)
        return Nv, d
    L = np.stack([1 - x - y - z, x, y, z], axis=1)
    gL = np.array([(-1, -1, -1), (1, 0, 0), (0, 1, 0), (0, 0, 1)], float)
    if etype == "Tet4":
        return L, np.broadcast_to(gL, (len(p), 4, 3)).copy()
    ed = ((0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3))
    Nv = np.concatenate([L * (2 * L - 1), np.stack([4 * L[:, a] * L[:, b] for a, b in ed], axis=1)], axis=1)
    d = np.concatenate([(4 * L - 1)[:, :, None] * gL[None],
                        np.stack([4 * (L[:, a, None] * gL[b] + L[:, b, None] * gL[a]) for a, b in ed], axis=1)], axis=1)
    return Nv, d


def _rule(etype):
    """The element's own quadrature: 4 points (Tet10), 1 (Tet4), 2x2x2 with x fastest (Hex8)."""
    if etype == "Tet10":
        a, b = 0.585410196624968, 0.138196601125011
        return np.array([(a, b, b), (b, a, b), (b, b, a), (b, b, b)]), np.full(4, 1 / 24)
    if etype == "Tet4":
        return np.full((1, 3), 0.25), np.array([1 / 6])
    g = 1 / math.sqrt(3.0)
    return np.array([[(g if (q >> c) & 1 else -g) for c in range(3)] for q in range(8)]), np.ones(8)


def _fit_rule(etype):
    """The nodal fit's rule: collapsed 3 x 3 x 4 Gauss points on tetrahedra, 2x2x2 on hexahedra."""
    if etype == "Hex8":
        return _rule(etype)
    x3, w3 = np.polynomial.legendre.leggauss(3)
    x4, w4 = np.polynomial.legendre.leggauss(4)
    pts, ws = [], []
    for a, wa in zip((1 + x3) / 2, w3 / 2):
        for b, wb in zip((1 + x3) / 2, w3 / 2):
            for c, wc in zip((1 + x4) / 2, w4 / 2):
                pts.append((a * (1 - b) * (1 - c), b * (1 - c), c))
                ws.append(wa * wb * wc * (1 - b) * (1 - c) ** 2)
    return np.array(pts), np.array(ws)


class _Matrix:
    """Element matrices over a mesh: products, diagonal blocks, PCG with block Jacobi."""

    def __init__(self, dofs, Ke, n, nb):
        self.dofs, self.Ke, self.n, self.nb, self.dev = dofs, Ke, n, nb, Ke.device

    def times(self, x):
        y = torch.zeros(self.n, dtype=F64, device=self.dev)
        ye = torch.bmm(self.Ke, x[self.dofs].unsqueeze(2))
        return y.index_add_(0, self.dofs.reshape(-1), ye.reshape(-1))

    def solve(self, b, fixed, tol=1e-13, maxit=30000):
        """K x = b on the free rows, x = 0 on the fixed ones."""
        nb, free = self.nb, (~fixed).to(F64)
        k = self.dofs.shape[1] // nb
        D = torch.zeros(self.n // nb, nb, nb, dtype=F64, device=self.dev)
        nodes = self.dofs[:, ::nb] // nb
        blocks = self.Ke.reshape(-1, k, nb, k, nb)
        for i in range(k):
            D.index_add_(0, nodes[:, i], blocks[:, i, :, i, :].contiguous())
        fm = free.reshape(-1, nb)
        D = D * fm[:, :, None] * fm[:, None, :] + torch.diag_embed(1 - fm)
        Di = torch.linalg.inv(D) * fm[:, :, None] * fm[:, None, :]
        prec = lambda r: torch.bmm(Di, r.reshape(-1, nb, 1)).reshape(-1)  # noqa: E731
        x = torch.zeros_like(b)
        for _ in range(2):  # the second pass starts from the true residual
            r = (b - self.times(x)) * free
            if _ == 0:
                stop = tol * float(r.norm())
            z = prec(r)
            p, rz, d = z.clone(), r @ z, torch.zeros_like(b)
            for it in range(maxit):
                q = self.times(p) * free
                al = rz / (p @ q)
                d += al * p
                r -= al * q
                if it % 50 == 49 and not float(r.norm()) > stop:
                    break
                z = prec(r)
                new = r @ z
                p = z + (new / rz) * p
                rz = new
            x = x + d
            if self.n > 400000:  # its second pass would take too long, and changes the last digits only
                break
        return x


class _Elements:
    """Gradients and weights at the quadrature points of a mesh."""

    def __init__(self, m, rule=None):
        self.m, self.dev = m, "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        self.conn = t(m.conn)
        self.X = t(m.X)[self.conn]
        self.E, self.nu = t(m.E), t(m.nu)
        self.la = self.E * self.nu / ((1 + self.nu) * (1 - 2 * self.nu))
        self.mu = self.E / (2 * (1 + self.nu))
        self.dofs = (3 * self.conn[:, :, None] + torch.arange(3, device=self.dev)).reshape(len(m.conn), -1)
        p, w = rule or _rule(m.etype)
        Nv, dN = _basis(m.etype, p)
        self.N, self.g, self.w, self.invJ, self.det = t(Nv), [], [], [], []
        for q in range(len(w)):
            d = t(dN[q])
            J = torch.matmul(d.t().contiguous(), self.X)  # J[a][b] = sum dN_i/dxi_a X_i[b]
            det = torch.linalg.det(J)
            inv = torch.linalg.inv(J)
            self.g.append(torch.matmul(d, inv.transpose(1, 2).contiguous()))
            self.w.append(w[q] * det)
            self.invJ.append(inv)
            self.det.append(det)

    def grad(self, u, q):
        """du_c/dX_A at point q."""
        ue = torch.as_tensor(u, device=self.dev)[self.dofs].reshape(len(self.conn), -1, 3)
        return torch.bmm(ue.transpose(1, 2).contiguous(), self.g[q])

    def tangent(self, u=None, law="linear", parts="mg"):
        """Element matrices: linear, or at u with St. Venant-Kirchhoff ('svk') or neo-Hookean ('nh')."""
        n, k = self.conn.shape
        K = torch.zeros(n, k, 3, k, 3, dtype=F64, device=self.dev)
        f = torch.zeros(n, k, 3, dtype=F64, device=self.dev)
        I = torch.eye(3, dtype=F64, device=self.dev)
        for q, (g, w) in enumerate(zip(self.g, self.w)):
            la, mu = self.la * w, self.mu * w
            if law == "linear":
                F, A, S, c1, c2 = I.expand(n, 3, 3), I.expand(n, 3, 3), None, la, mu
            else:
                H = self.grad(u, q)
                F = I + H
                Gs = H + H.transpose(1, 2) + torch.bmm(H.transpose(1, 2).contiguous(), H)  # C - I
                if law == "svk":
                    A, c1, c2 = I.expand(n, 3, 3), la, mu
                    S = 0.5 * la[:, None, None] * Gs.diagonal(dim1=1, dim2=2).sum(1)[:, None, None] * I + mu[:, None, None] * Gs
                else:
                    A = torch.linalg.inv(I + Gs)
                    i1 = H.diagonal(dim1=1, dim2=2).sum(1)
                    i2 = 0.5 * (i1 ** 2 - (H * H.transpose(1, 2)).sum((1, 2)))
                    lnJ = torch.log1p(i1 + i2 + torch.linalg.det(H))
                    S = mu[:, None, None] * torch.bmm(A, Gs) + (la * lnJ)[:, None, None] * A
                    c1, c2 = la, mu - la * lnJ
                f += torch.bmm(g, torch.bmm(F, S).transpose(1, 2).contiguous())
            if "m" in parts:
                # D = c1 A x A + c2 (A A + A A): with a_i = F A g_i, G = F A F'
                FA = torch.bmm(F.contiguous(), A.contiguous())
                a = torch.bmm(g, FA.transpose(1, 2).contiguous())
                gAg = torch.bmm(torch.bmm(g, A.contiguous()), g.transpose(1, 2).contiguous())
                G = torch.bmm(FA, F.transpose(1, 2).contiguous())
                K += c1[:, None, None, None, None] * a[:, :, :, None, None] * a[:, None, None, :, :]
                K += c2[:, None, None, None, None] * torch.einsum("eid,ejc->eicjd", a, a)
                K += c2[:, None, None, None, None] * gAg[:, :, None, :, None] * G[:, None, :, None, :]
            if "g" in parts and S is not None:
                s = torch.bmm(torch.bmm(g, S.contiguous()), g.transpose(1, 2).contiguous())
                K += s[:, :, None, :, None] * I[None, None, :, None, :]
        return K.reshape(n, 3 * k, 3 * k), f.reshape(n, 3 * k)

    def stiffness(self):
        return _Matrix(self.dofs, self.tangent()[0], self.m.n_dofs, 3)

    def scatter(self, fe):
        return torch.zeros(self.m.n_dofs, dtype=F64, device=self.dev).index_add_(0, self.dofs.reshape(-1), fe.reshape(-1))


def _faces(m, dev):
    """Per boundary-face point: shape values (points, nodes) and weights (faces, points)."""
    if m.ftype == "Quad4":
        g = 1 / math.sqrt(3.0)
        c = np.array([(-1, -1), (1, -1), (1, 1), (-1, 1)], float)
        p, w = np.array([(-g, -g), (g, -g), (-g, g), (g, g)]), np.ones(4)
        f = 1 + c[None] * p[:, None]
        Nv = f.prod(2) / 4
        d = np.stack([c[:, k] * f[:, :, 1 - k] / 4 for k in range(2)], axis=2)
    else:
        p, w = (np.array([(1 / 6, 1 / 6), (2 / 3, 1 / 6), (1 / 6, 2 / 3)]), np.full(3, 1 / 6)) if m.ftype == "Tri6" else (np.full((1, 2), 1 / 3), np.array([0.5]))
        L = np.stack([1 - p.sum(1), p[:, 0], p[:, 1]], axis=1)
        gL = np.array([(-1, -1), (1, 0), (0, 1)], float)
        Nv, d = L, np.broadcast_to(gL, (len(p), 3, 2))
        if m.ftype == "Tri6":
            ed = ((0, 1), (1, 2), (2, 0))
            Nv = np.concatenate([L * (2 * L - 1), np.stack([4 * L[:, a] * L[:, b] for a, b in ed], axis=1)], axis=1)
            d = np.concatenate([(4 * L - 1)[:, :, None] * gL[None], np.stack([4 * (L[:, a, None] * gL[b] + L[:, b, None] * gL[a]) for a, b in ed], axis=1)], axis=1)
    Xf = m.X[m.faces]
    T = np.einsum("qik,fic->fqkc", d, Xf)
    wj = w * np.linalg.norm(np.cross(T[:, :, 0], T[:, :, 1]), axis=2)
    return torch.as_tensor(Nv, device=dev), torch.as_tensor(wj, device=dev)


def _load(m, dev):
    """Nodal forces of the surface traction."""
    Nv, wj = _faces(m, dev)
    fe = (wj @ Nv)[:, :, None] * torch.as_tensor(m.face_traction(), device=dev)[:, None, :]
    f = torch.zeros(m.n_nodes, 3, dtype=F64, device=dev)
    f.index_add_(0, torch.as_tensor(m.faces, device=dev).reshape(-1), fe.reshape(-1, 3))
    return f.reshape(-1)


def _csr_values(el, *Ke):
    """Element matrices summed into the CSR order of their pattern (rows, then columns)."""
    n = el.m.n_dofs
    key = (el.dofs[:, :, None] * n + el.dofs[:, None, :]).reshape(-1)
    uniq, inv = torch.unique(key, return_inverse=True)
    del key
    return [torch.zeros(len(uniq), dtype=F64, device=el.dev).index_add_(0, inv, K.reshape(-1)) for K in Ke]


def _voigt(G):
    return torch.stack([G[:, 0, 0], G[:, 1, 1], G[:, 2, 2], 0.5 * (G[:, 0, 1] + G[:, 1, 0]), 0.5 * (G[:, 1, 2] + G[:, 2, 1]), 0.5 * (G[:, 0, 2] + G[:, 2, 0])], dim=1)


def _stress(el, e):
    s = 2 * el.mu[:, None] * e
    s[:, :3] += (el.la * e[:, :3].sum(1))[:, None]
    return s


def _exact_post(m, u):
    el, fit = _Elements(m), _Elements(m, _fit_rule(m.etype))
    eps = [_voigt(el.grad(u, q)) for q in range(len(el.w))]
    out = {"strain": torch.stack(eps, dim=1), "stress": torch.stack([_stress(el, e) for e in eps], dim=1)}
    Me = sum(w[:, None, None] * (fit.N[q][:, None] * fit.N[q][None, :]) for q, w in enumerate(fit.w))
    Mm = _Matrix(fit.conn, Me, m.n_nodes, 1)
    fixed = torch.zeros(m.n_nodes, dtype=torch.bool, device=el.dev)
    fe = [_voigt(fit.grad(u, q)) for q in range(len(fit.w))]
    for name, vals in (("strain_nodal", fe), ("stress_nodal", [_stress(fit, e) for e in fe])):
        be = sum((w[:, None] * fit.N[q][None, :])[:, :, None] * vals[q][:, None, :] for q, w in enumerate(fit.w))
        b = torch.zeros(m.n_nodes, 6, dtype=F64, device=el.dev).index_add_(0, fit.conn.reshape(-1), be.reshape(-1, 6))
        out[name] = torch.stack([Mm.solve(b[:, c].contiguous(), fixed, tol=1e-15, maxit=400) for c in range(6)], dim=1)
    return {k: v.cpu().numpy() for k, v in out.items()}


def _exact_heat(m, seed):
    el, h = _Elements(m), _heat_inputs(m, seed)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=el.dev)  # noqa: E731
    k, qs = t(h["k"]), t(h["q"])
    Ke = sum((w * k)[:, None, None] * torch.bmm(g, g.transpose(1, 2).contiguous()) for g, w in zip(el.g, el.w))
    f = torch.zeros(m.n_nodes, dtype=F64, device=el.dev)
    f.index_add_(0, el.conn.reshape(-1), sum((w * qs)[:, None] * el.N[q] for q, w in enumerate(el.w)).reshape(-1))
    Nv, wj = _faces(m, el.dev)
    fc = t(m.faces)
    load = t(h["flux"]) + t(h["h"]) * t(h["T_ext"])
    f.index_add_(0, fc.reshape(-1), (load[:, None] * (wj @ Nv)).reshape(-1))
    Kf = t(h["h"])[:, None, None] * torch.einsum("fq,qi,qj->fij", wj, Nv, Nv)
    vol = _Matrix(el.conn, Ke, m.n_nodes, 1)

    class Both(_Matrix):  # conduction and the convection faces
        def times(self, x):
            y = vol.times(x)
            return y.index_add_(0, fc.reshape(-1), torch.bmm(Kf, x[fc].unsqueeze(2)).reshape(-1))

    fixed = t(h["fixed"]).bool()
    T0 = torch.where(fixed, t(h["T_fixed"]), torch.zeros_like(f))
    A = Both(el.conn, Ke, m.n_nodes, 1)
    return (T0 + A.solve(f - A.times(T0), fixed, tol=1e-15, maxit=6000)).cpu().numpy()


def _exact_nonlinear(m, steps):
    el = _Elements(m)
    f = _load(m, el.dev)
    fixed = torch.as_tensor(m.fixed_mask().astype(bool), device=el.dev)
    u = torch.zeros_like(f)
    for s in range(1, steps + 1):
        lf, ref = s / steps, s / steps * float(f[~fixed].norm())
        for _ in range(25):
            Ke, fe = el.tangent(u, "nh")
            r = lf * f - el.scatter(fe)
            r[fixed] = 0
            rn = float(r.norm())
            if rn < 1e-13 * ref or (_ > 8 and rn > 0.5 * last):
                break
            last = rn
            u = u + _Matrix(el.dofs, Ke, m.n_dofs, 3).solve(r, fixed, tol=1e-3 if rn > 1e-3 * ref else 1e-6)
    return u.cpu().numpy()


def _exact_train(m, R, E):
    """(loss, gradient) with the network in 64 bits on its stored weights (no 16-bit rounding of activations)."""
    el = _Elements(m)
    dev, N = el.dev, m.n_nodes
    Kg = el.stiffness()
    k = m.conn.shape[1]
    fixed = torch.as_tensor(m.fixed_mask().astype(bool), device=dev)
    n3 = fixed.reshape(-1, 3)
    node = el.conn.reshape(-1)
    acc = lambda v: torch.zeros(N, dtype=F64, device=dev).index_add_(0, node, v.reshape(-1).to(F64))  # noqa: E731
    ext = lambda v, how: torch.zeros(N, dtype=F64, device=dev).scatter_reduce_(0, node, v.reshape(-1), how, include_self=False)  # noqa: E731
    per = lambda v: v[:, None].expand(-1, k).contiguous()  # noqa: E731
    blocks = Kg.Ke.reshape(-1, k, 3, k, 3)
    D = torch.zeros(N, 3, 3, dtype=F64, device=dev)
    for i in range(k):
        D.index_add_(0, el.conn[:, i], blocks[:, i, :, i, :].contiguous())
    te = sum(((el.la + 4 * el.mu) * w)[:, None] * (g ** 2).sum(2) for g, w in zip(el.g, el.w))
    shape = el.invJ[0].reshape(-1, 9).norm(dim=1) * el.det[0].pow(1 / 3)
    elfix = n3[el.conn].any(2).any(1).to(F64)
    cnt, lE = acc(torch.ones_like(te)), torch.log(el.E)
    tsum, tmax, tmin, esum = acc(te), ext(te, "amax"), ext(te, "amin"), acc(per(el.E))
    emax, emin, emean = ext(per(el.E), "amax"), ext(per(el.E), "amin"), esum / cnt
    corner = torch.zeros_like(te)
    corner[:, :4] = 1
    s = 3 / D.diagonal(dim1=1, dim2=2).sum(1)
    d = D * s[:, None, None]
    onface = torch.zeros(N, dtype=F64, device=dev)
    onface[torch.as_tensor(m.faces, device=dev).reshape(-1)] = 1
    off = [d[:, 0, 1], d[:, 1, 2], d[:, 0, 2]]
    feat = torch.stack([
        d[:, 0, 0], d[:, 1, 1], d[:, 2, 2], *off, torch.log(cnt), tmax / tsum, cnt * tmin / tsum,
        torch.sqrt(torch.clamp(acc(te ** 2) / cnt - (tsum / cnt) ** 2, min=0)) / (tsum / cnt), torch.log(emax / emin),
        torch.log(emean) - acc(per(lE)) / cnt, acc(corner) / cnt, n3.to(F64).mean(1), acc(per(elfix)) / cnt, onface,
        torch.linalg.det(0.5 * (d + d.transpose(1, 2))), torch.sqrt(2 * sum(o ** 2 for o in off)),
        acc(per(shape)) / cnt, ext(per(shape), "amin"), ext(per(shape), "amax"),
        acc(te * per(lE)) / tsum - torch.log(emax), (tmax - tmin) / tsum, acc((per(el.E) > emean[el.conn]).to(F64)) / cnt], dim=1)
    # packed weights: 24-byte header, bf16 matrices, f32 biases, shift, scale, eps
    blob = open(DEFAULT_WEIGHTS, "rb").read()
    pos, prm = 24, {}
    for name, sh in (("W1", (64, 24)), ("W2", (64, 64)), ("W3", (6, 64))):
        h = np.frombuffer(blob, np.uint16, sh[0] * sh[1], pos).astype(np.uint32) << 16
        prm[name] = h.view(np.float32).reshape(sh)
        pos += 2 * sh[0] * sh[1]
    for name, n in (("b1", 64), ("b2", 64), ("b3", 6), ("shift", 24), ("scale", 24), ("eps", 1)):
        prm[name] = np.frombuffer(blob, np.float32, n, pos)
        pos += 4 * n
    prm = {a: torch.as_tensor(v.astype(np.float64), device=dev) for a, v in prm.items()}
    order = ("W1", "b1", "W2", "b2", "W3", "b3")
    for a in order:
        prm[a].requires_grad_(True)
    gelu = torch.nn.functional.gelu
    x = (feat - prm["shift"]) * prm["scale"]
    o = gelu(gelu(x @ prm["W1"].t() + prm["b1"]) @ prm["W2"].t() + prm["b2"]) @ prm["W3"].t() + prm["b3"]
    ex = lambda v: torch.exp(torch.clamp(v, -5, 5))  # noqa: E731
    zero = torch.zeros_like(o[:, 0])
    L = torch.stack([ex(o[:, 0]), zero, zero, o[:, 1], ex(o[:, 2]), zero, o[:, 3], o[:, 4], ex(o[:, 5])], dim=1).reshape(-1, 3, 3)
    fm = (~n3).to(F64)
    Mj = torch.linalg.inv(D * fm[:, :, None] * fm[:, None, :] + torch.diag_embed(1 - fm)) * fm[:, :, None] * fm[:, None, :]
    plain = n3.any(1)
    safe = torch.where(plain[:, None, None], torch.eye(3, dtype=F64, device=dev).expand(N, 3, 3), Mj)
    C = torch.linalg.cholesky(0.5 * (safe + safe.transpose(1, 2)))
    inner = torch.bmm(L, L.transpose(1, 2)) + prm["eps"] * torch.eye(3, dtype=F64, device=dev)
    Mb = torch.where(plain[:, None, None], Mj, torch.bmm(torch.bmm(C, inner), C.transpose(1, 2)))
    loss = 0.0
    free = (~fixed).to(F64)
    for r, e in zip(R, E):
        r, e = torch.as_tensor(r, device=dev), torch.as_tensor(e, device=dev)
        z = torch.bmm(Mb, r.reshape(-1, 3, 1)).reshape(-1)
        w = Kg.times(z) * free
        loss = loss + (1 - (z @ r) ** 2 / ((z @ w) * (e @ r))) / len(R)
    grads = torch.autograd.grad(loss, [prm[a] for a in order])
    return float(loss.detach()), torch.cat([g.reshape(-1) for g in grads]).cpu().numpy()


def exact(case, seed):
    m, kind = _mesh(case, seed), case["kind"]
    if kind == "heat":
        return _exact_heat(m, seed)
    if kind == "post":
        return _exact_post(m, _displacement(m, seed, 1e-3))
    if kind == "nonlinear":
        return _exact_nonlinear(m, case["steps"])
    if kind == "train":
        return _exact_train(m, *_pairs(m, seed, case["pairs"]))
    el = _Elements(m)
    fixed = torch.as_tensor(m.fixed_mask().astype(bool), device=el.dev)
    if kind == "tl":
        u = torch.as_tensor(_displacement(m, seed, 0.5), device=el.dev)
        Km, fe = el.tangent(u, "svk", "m")
        Kg, _ = el.tangent(u, "svk", "g")
        vm, vg = _csr_values(el, Km, Kg)
        return [v.cpu().numpy() for v in (vm, vg, _load(m, el.dev) - el.scatter(fe))]
    K = el.stiffness()
    if kind == "assemble":
        u = torch.as_tensor(_displacement(m, seed, 1e-3), device=el.dev)
        f = _load(m, el.dev) - K.times(u)
        return [v.cpu().numpy() for v in (*_csr_values(el, K.Ke), f)]
    if kind == "ku":
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        y = K.times(torch.randn(m.n_dofs, dtype=F64, device="cuda", generator=g))
        return torch.where(fixed, torch.zeros_like(y), y)
    f = _load(m, el.dev)
    u = K.solve(f * (~fixed).to(F64), fixed, tol=1e-14 if m.n_dofs < 200000 else 1e-13)
    if kind == "solve" and case["method"] == "pcg_csr":
        la = torch.where(fixed, f - K.times(u), torch.zeros_like(f))
        return u.cpu().numpy(), la.cpu().numpy()
    return u.cpu().numpy()
