"""The resident PCG (persist.hip), through the C ABI.

Meshes at the edges of its patches (128 Tet10 or 512 Tet4 elements), of its
groups of 16 workgroups and of its range (256 workgroups), against the oracle's
direct solve, and against the launched iterations (JFEM_PERSIST=0, a child
process): the FP64 iteration counts differ only by the order of the reductions
(3% + 2; the FP32 inner solves restart at FP32's attainable residual, where
rounding decides the count), the answers are bit-reproducible.  Heat conduction (convection faces
on elements, and one that is on none) and the nodal fits run resident too.  The
bars follow from the solves' own tolerance: the residual 1e-10 (1e-11 is below what the FP64
residual of such a cantilever can show) bounds the error at 1e-8 for these meshes
(the direct solve itself is good to 1e-10).
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from jfem import mesh as M

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# name -> (generator, grid); workgroups in the comments
CASES = {
    "tet10_6": ("box_tet10", (1, 1, 1)),        # 1, six elements
    "tet10_126": ("box_tet10", (7, 3, 1)),      # 1, two elements short of a patch
    "tet10_132": ("box_tet10", (11, 2, 1)),     # 2, four elements in the second
    "tet10_2016": ("box_tet10", (14, 6, 4)),    # 16, one group
    "tet10_2052": ("box_tet10", (19, 6, 3)),    # 17, two groups, the second of one
    "tet4_510": ("box_tet4", (17, 5, 1)),       # 1
    "tet4_10368": ("box_tet4", (24, 9, 8)),     # 21
}
_CHILD = r"""
import json, sys
sys.path[:0] = [{pkg!r}]
import jfem
from jfem import mesh as M
out = {{}}
for name, (gen, g) in json.loads({cases!r}).items():
    m = getattr(M, gen)(*g, seed=5, jitter=0.1, E_sigma=0.4)
    c = jfem.Context(0)
    c.upload(m)
    for meth in (0, 1):
        print("launched", name, meth, flush=True)
        out[f"{{name}}/{{meth}}"] = c.solve(method=meth, rtol=1e-10, inner_rtol=1e-2)[2]["iterations"]
    c.close()
json.dump(out, open({out!r}, "w"))
"""


def say(msg):
    print(f"[gpu] {msg}", flush=True)


@pytest.fixture(scope="module")
def launched(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("launched") / "it.json")
    code = _CHILD.format(pkg=os.path.join(ROOT, "juliafem.jl_amd"), cases=json.dumps(CASES), out=out)
    subprocess.run([sys.executable, "-c", code], env=dict(os.environ, JFEM_PERSIST="0"), check=True, timeout=120)
    return json.load(open(out))


@pytest.mark.parametrize("name", list(CASES))
def test_resident_pcg(oracle, launched, name):
    import jfem
    gen, g = CASES[name]
    m = getattr(M, gen)(*g, seed=5, jitter=0.1, E_sigma=0.4)
    csr = oracle.assemble_csr(m)
    ud, _, _ = oracle.solve_direct_lapack(csr, m.fixed_mask(), np.zeros(m.n_dofs), oracle.load_vector(m))
    ctx = jfem.Context(0)
    ctx.upload(m)
    for meth in (0, 1):   # FP64 PCG; FP32 PCG in FP64 refinement
        say(f"resident {name} method={meth} nodes={m.n_nodes} el={m.n_el}")
        u, _, st = ctx.solve(method=meth, rtol=1e-10, inner_rtol=1e-2)
        u2, _, _ = ctx.solve(method=meth, rtol=1e-10, inner_rtol=1e-2)
        assert np.array_equal(u, u2)
        assert np.linalg.norm(u - ud) <= 1e-8 * np.linalg.norm(ud)
        it = launched[f"{name}/{meth}"]
        if meth == 1 or it > m.n_dofs - 3 * len(m.clamp_nodes):
            continue   # past CG's exact termination the count is rounding alone
        assert abs(st["iterations"] - it) <= 2 + 0.03 * it
    ctx.close()


def test_resident_edges(oracle):
    """Iteration cap, a zero load, prescribed displacements, user blocks and a
    given right-hand side behave as in the launched form."""
    import jfem
    m = M.box_tet10(12, 3, 3, seed=8, jitter=0.1, E_sigma=0.4)
    csr = oracle.assemble_csr(m)
    ctx = jfem.Context(0)
    ctx.upload(m)
    say("iteration cap")
    u, _, st = ctx.solve(rtol=1e-10, maxit=7, raise_on_noconv=False)
    assert st["iterations"] == 7 and st["converged"] == 0 and np.all(np.isfinite(u))
    say("zero load")
    u, _, st = ctx.solve(f=np.zeros(m.n_dofs))
    assert not np.any(u) and st["iterations"] == 0
    say("user blocks")
    blocks = np.tile(np.eye(3).ravel(), (m.n_nodes, 1)) * 1e-4
    ctx.set_preconditioner_blocks(blocks)
    f = oracle.load_vector(m) * 3.0
    u, la, _ = ctx.solve(f=f, precond=2, rtol=1e-10, maxit=100000, want_la=True)
    ud, lad, _ = oracle.solve_direct_lapack(csr, m.fixed_mask(), np.zeros(m.n_dofs), f)
    assert np.linalg.norm(u - ud) <= 1e-8 * np.linalg.norm(ud)
    say("prescribed displacements")
    g = np.zeros(m.n_dofs)
    g[3 * m.clamp_nodes + 2] = 1e-3
    ctx.upload_bcs(m.fixed_mask(), g, m.faces, m.ftype, m.face_traction())
    u, la, _ = ctx.solve(rtol=1e-10, want_la=True)
    ud, lad, _ = oracle.solve_direct_lapack(csr, m.fixed_mask(), g, oracle.load_vector(m))
    assert np.linalg.norm(u - ud) <= 1e-8 * np.linalg.norm(ud)
    ctx.close()


# elements per patch: Tet10 128, Hex8 256, Tet4 512
OTHER = [("box_tet10", (7, 3, 1)), ("box_tet10", (19, 6, 3)), ("box_hex8", (17, 5, 3)), ("box_hex8", (37, 7, 1)),
         ("box_tet4", (24, 9, 8))]


@pytest.mark.parametrize("gen,g", OTHER)
@pytest.mark.parametrize("attached", [True, False])
def test_resident_heat(oracle, gen, g, attached):
    """Bar: rtol 1e-12 on the residual, 1e-8 on the temperatures, as the heat
    tests of one patch ask."""
    import jfem
    m = getattr(M, gen)(*g, seed=6, jitter=0.1)
    rng = np.random.default_rng(3)
    k, q = np.exp(0.5 * rng.standard_normal(m.n_el)) * 3.0, rng.uniform(0.5, 2.0, m.n_el)
    faces = m.faces.copy()
    if not attached:   # a face whose nodes no element holds together
        faces[0] = np.linspace(0, m.n_nodes - 1, faces.shape[1]).astype(np.int64)
    nf = faces.shape[0]
    flux, h, te = rng.uniform(0, 1, nf), rng.uniform(0.5, 1.0, nf), rng.uniform(10, 20, nf)
    fixed = np.isclose(m.X[:, 0], 0.0)
    Tf = np.full(m.n_nodes, 5.0)
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"resident heat {gen} {g} attached={attached}")
    T, st = ctx.heat_solve(k, q, faces, flux=flux, h=h, T_ext=te, fixed=fixed, T_fixed=Tf, rtol=1e-12)
    Kh, f = oracle.heat_system(m, k, q=q, faces=faces, ftype=m.ftype, flux=flux, h=h, T_ext=te)
    To = oracle.heat_solve_direct(Kh, f, fixed, Tf)
    assert st["converged"] == 1
    assert np.abs(T - To).max() <= 1e-8 * np.abs(To).max()
    ctx.close()


@pytest.mark.parametrize("gen,g", OTHER)
def test_resident_fit(oracle, gen, g):
    """Bar: 1e-9 of the largest value, as the fit tests of one patch ask."""
    import jfem
    m = getattr(M, gen)(*g, seed=6, jitter=0.1)
    u = np.random.default_rng(4).standard_normal(m.n_dofs) * 1e-3
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"resident fit {gen} {g}")
    out = ctx.postprocess(u)
    one = ctx.postprocess(u, gauss=False)
    for field in ("strain", "stress"):
        ref = oracle.lsq_fit(m, u, field)
        assert np.abs(out[field + "_nodal"] - ref).max() <= 1e-9 * np.abs(ref).max()
        assert np.array_equal(out[field + "_nodal"], one[field + "_nodal"])
    ctx.close()


@pytest.mark.parametrize("name,coarse_nodes", [("tet10_6", 64), ("tet10_132", 1000000), ("tet10_2016", 40),
                                               ("tet10_2052", 300), ("tet4_10368", 200)])
def test_resident_two_level(oracle, name, coarse_nodes):
    """The coarse correction in the resident PCG: one aggregate for the whole
    mesh, many in one patch and aggregates over several patches, to the bars of
    test_resident_pcg."""
    import jfem
    gen, g = CASES[name]
    m = getattr(M, gen)(*g, seed=5, jitter=0.1, E_sigma=0.4)
    csr = oracle.assemble_csr(m)
    ud, _, _ = oracle.solve_direct_lapack(csr, m.fixed_mask(), np.zeros(m.n_dofs), oracle.load_vector(m))
    ctx = jfem.Context(0)
    ctx.upload(m)
    for meth in (0, 1):
        say(f"resident two-level {name} method={meth} coarse_nodes={coarse_nodes}")
        kw = dict(method=meth, rtol=1e-10, inner_rtol=1e-2, coarse_nodes=coarse_nodes)
        u, _, _ = ctx.solve(**kw)
        assert np.linalg.norm(u - ud) <= 1e-8 * np.linalg.norm(ud)
        assert np.array_equal(u, ctx.solve(**kw)[0])
    ctx.close()


@pytest.mark.parametrize("name", ["tet10_6", "tet10_132", "tet10_2052"])
@pytest.mark.parametrize("coarse_nodes", [0, 100])
def test_resident_tangent(oracle, name, coarse_nodes):
    """The neo-Hookean tangent in the resident PCG against the oracle's Newton
    with direct tangent solves: 1e-7, as the nonlinear tests ask."""
    import jfem
    gen, g = CASES[name]
    m = getattr(M, gen)(*g, seed=5, jitter=0.1, E_sigma=0.4, traction=(0.0, 0.0, -2.0))
    uo, _ = oracle.nh_newton(m, load_steps=1, rtol=1e-10)
    ctx = jfem.Context(0)
    ctx.upload(m)
    for meth in (0, 1):
        say(f"resident tangent {name} method={meth} coarse_nodes={coarse_nodes}")
        kw = dict(load_steps=1, rtol=1e-10, method=meth, coarse_nodes=coarse_nodes)
        u, st = ctx.solve_nonlinear(**kw)
        assert st["converged"] == 1
        assert np.linalg.norm(u - uo) <= 1e-7 * np.linalg.norm(uo)
        assert np.array_equal(u, ctx.solve_nonlinear(**kw)[0])
    ctx.close()


# nodes: 27 (one workgroup), 2,016 (63, four groups), 3,451, 2,250; 10,496 nodes: 41 of each
# of 256 workgroups, also in random order (long lists of other workgroups' nodes)
CSR = {"tet10_6": CASES["tet10_6"], "hex8_1435": ("box_hex8", (41, 5, 7)), "tet10_2052": CASES["tet10_2052"],
       "tet4_10368": CASES["tet4_10368"], "hex8_9000": ("box_hex8", (40, 15, 15)), "hex8_9000_shuffled": ("box_hex8", (40, 15, 15))}


@pytest.mark.parametrize("name", list(CSR))
def test_resident_csr(oracle, name):
    """The assembled matrix in the resident PCG against the oracle's direct solve,
    or against the matrix-free solve where that is too large: a hundred times the
    solve's tolerance, as above.  That is 1e-9 here: the FP64 residual with this
    matrix ends at 1.0e-10 to 2.2e-10, launched or resident."""
    import jfem
    gen, g = CSR[name]
    m = getattr(M, gen)(*g, seed=5, jitter=0.1, E_sigma=0.4)
    if "shuffled" in name:
        m = M.renumber(m, np.random.default_rng(1).permutation(m.n_nodes))
    ctx = jfem.Context(0)
    ctx.upload(m)
    if m.n_dofs < 12000:
        ud, lad, _ = oracle.solve_direct_lapack(oracle.assemble_csr(m), m.fixed_mask(), np.zeros(m.n_dofs), oracle.load_vector(m))
    else:
        ud, lad, _ = ctx.solve(op="matfree", rtol=1e-10, want_la=True)
    for meth in (0, 1):
        say(f"resident csr {name} method={meth} nodes={m.n_nodes}")
        kw = dict(op="csr", method=meth, rtol=1e-9, inner_rtol=1e-2, want_la=True)
        u, la, _ = ctx.solve(**kw)
        assert np.linalg.norm(u - ud) <= 1e-7 * np.linalg.norm(ud)
        u2, la2, _ = ctx.solve(**kw)
        assert np.array_equal(u, u2) and np.array_equal(la, la2)
    ctx.close()


# 256 elements per patch: one element, one short of a patch, a full one, two, 18
@pytest.mark.parametrize("g", [(1, 1, 1), (17, 5, 3), (16, 4, 4), (13, 5, 4), (40, 11, 10)])
@pytest.mark.parametrize("jitter", [0.0, 0.15])
def test_resident_hex8(oracle, g, jitter):
    """Hex8 elasticity, parallelepipeds and general hexahedra, one-level and
    two-level, to the bars of test_resident_pcg (the larger mesh, whose residual
    ends above 1e-10, at ten times both)."""
    import jfem
    m = M.box_hex8(*g, L=(4.0, 4.0 * g[1] / g[0], 4.0 * g[2] / g[0]), seed=5, jitter=jitter, E_sigma=0.4)
    k = 10.0 if m.n_el > 4000 else 1.0
    csr = oracle.assemble_csr(m)
    ud, _, _ = oracle.solve_direct_lapack(csr, m.fixed_mask(), np.zeros(m.n_dofs), oracle.load_vector(m))
    ctx = jfem.Context(0)
    ctx.upload(m)
    for meth in (0, 1):
        for coarse_nodes in (0, 100):
            say(f"resident hex8 {g} jitter={jitter} method={meth} coarse_nodes={coarse_nodes}")
            kw = dict(method=meth, rtol=k * 1e-10, inner_rtol=1e-2, coarse_nodes=coarse_nodes)
            u, _, _ = ctx.solve(**kw)
            assert np.linalg.norm(u - ud) <= k * 1e-8 * np.linalg.norm(ud)
            assert np.array_equal(u, ctx.solve(**kw)[0])
    ctx.close()


@pytest.mark.parametrize("whose", ["none", "wedge"])
def test_heat_face_at_a_collapsed_hex(oracle, whose):
    """A wedge (a Hex8 with two of its nodes twice): a convection face of four nodes
    of which it has three, one of them twice (no element's face), and one of its own
    with both doubled nodes.  Bars as test_resident_heat."""
    import jfem
    b = M.box_hex8(4, 3, 2, seed=6, jitter=0.05)
    conn = b.conn.copy()
    w = conn[0].copy()          # its edges 2-6 onto 1-5: the wedge 0 1 3, 4 5 7
    w[2], w[6] = w[1], w[5]
    conn[0] = w
    used, conn = np.unique(conn, return_inverse=True)
    m = M.Mesh(X=b.X[used], conn=conn.reshape(-1, 8), etype="Hex8", E=b.E, nu=b.nu, faces=np.zeros((0, 4), np.int64),
               ftype="Quad4", clamp_nodes=np.zeros(0, np.int64))
    c = m.conn[0]
    far = int(m.conn[-1].max())
    assert len(set(c)) == 6 and far not in c
    faces = np.array([[c[1], c[3], c[0], far] if whose == "none" else [c[0], c[1], c[5], c[4]], m.conn[-1][4:]], np.int64)
    rng = np.random.default_rng(3)
    k, q = np.exp(0.5 * rng.standard_normal(m.n_el)) * 3.0, rng.uniform(0.5, 2.0, m.n_el)
    flux, h, te = rng.uniform(0, 1, 2), rng.uniform(0.5, 1.0, 2), rng.uniform(10, 20, 2)
    fixed = np.isclose(m.X[:, 0], m.X[:, 0].max())
    Tf = np.full(m.n_nodes, 5.0)
    ctx = jfem.Context(0)
    ctx.upload_mesh(m.X, m.conn, m.etype, m.E, m.nu)
    say(f"heat, a face at a collapsed hex: {whose}")
    T, st = ctx.heat_solve(k, q, faces, flux=flux, h=h, T_ext=te, fixed=fixed, T_fixed=Tf, rtol=1e-12)
    Kh, f = oracle.heat_system(m, k, q=q, faces=faces, ftype="Quad4", flux=flux, h=h, T_ext=te)
    To = oracle.heat_solve_direct(Kh, f, fixed, Tf)
    assert st["converged"] == 1
    assert np.abs(T - To).max() <= 1e-8 * np.abs(To).max()
    ctx.close()
