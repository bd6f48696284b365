"""The same call gives the same bits whatever was called before it (include/jfem.h),
through the C ABI.

A product jfm_apply, a training gradient or an assembly on the same mesh lies
between two equal solves (and two equal assemblies), with prescribed
displacements, so that the right-hand side, the FP64 residuals and the reactions
all take products with K; on meshes whose iterations run resident and on meshes
that turn out not to fit (a node of no element, more coarse unknowns than the
resident form holds).  Compared bit for bit.
"""
import numpy as np
import pytest

from jfem import mesh as M

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu] {msg}", flush=True)


def with_orphan(m):
    X = np.vstack([m.X, m.X.mean(0) + 0.01])
    return M.Mesh(X=X, conn=m.conn, etype=m.etype, E=m.E, nu=m.nu, faces=m.faces, ftype=m.ftype,
                  clamp_nodes=np.append(m.clamp_nodes, len(X) - 1), traction=m.traction)


TET10 = lambda: M.box_tet10(14, 6, 4, seed=5, jitter=0.1, E_sigma=0.4)  # 2,016 elements, 3,393 nodes
CASES = {
    "tet10": (TET10, 0), "hex8": (lambda: M.box_hex8(17, 5, 3, seed=5, jitter=0.1, E_sigma=0.4), 0),
    "tet10_two_level": (TET10, 200),
    "tet10_coarse_too_large": (TET10, 10),          # more than 256 aggregates
    "tet10_orphan": (lambda: with_orphan(TET10()), 0),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("method", [0, 1])
def test_solve_between_other_calls(name, method):
    import jfem
    make, coarse_nodes = CASES[name]
    m = make()
    ctx = jfem.Context(0)
    ctx.upload(m)
    rng = np.random.default_rng(7)
    g = np.zeros(m.n_dofs)
    g[3 * m.clamp_nodes + 1] = rng.normal(0.0, 1e-3, len(m.clamp_nodes))
    ctx.upload_bcs(m.fixed_mask(), g, m.faces, m.ftype, m.face_traction())
    x = rng.normal(0.0, 1e-3, m.n_dofs)
    kw = dict(method=method, rtol=1e-9, inner_rtol=1e-2, coarse_nodes=coarse_nodes, want_la=True, raise_on_noconv=False)
    say(f"solve, apply, solve: {name} method={method} nodes={m.n_nodes} el={m.n_el}")
    f0 = ctx.assemble(x)[1]
    u, la, st = ctx.solve(**kw)
    y = ctx.apply(x)
    for between in (lambda: ctx.apply(x), lambda: ctx.solve(op="csr", op_outer="csr", rtol=1e-6, raise_on_noconv=False)):
        between()
        u2, la2, st2 = ctx.solve(**kw)
        assert np.array_equal(u, u2) and np.array_equal(la, la2)
        assert st["iterations"] == st2["iterations"] and st["relres"] == st2["relres"]
    assert np.array_equal(ctx.assemble(x)[1], f0)
    assert np.array_equal(ctx.apply(x), y)
    ctx.close()
