"""Which solves run in a resident kernel (persist.hip, persist_csr.hip), and what
becomes of those whose waits give up, through the C ABI.

JFEM_PERSIST_POLLS bounds every wait of the resident kernels to that many looks:
with 0 the first exchange gives up, with a few some later one; every kernel ends
by itself, and the solve is repeated with launched iterations.  Results keep the
bars of the resident PCG's tests (1e-8 of the direct solve at rtol 1e-10, 1e-7
for Newton, 1e-9 for the nodal fits).
"""
import threading

import numpy as np
import pytest

from jfem import mesh as M

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu] {msg}", flush=True)


def box():
    return M.box_tet10(19, 6, 3, seed=5, jitter=0.1, E_sigma=0.4)   # 2,052 elements: 17 workgroups


@pytest.fixture(scope="module")
def direct(oracle):
    m = box()
    f = oracle.load_vector(m)
    return oracle.solve_direct_lapack(oracle.assemble_csr(m), m.fixed_mask(), np.zeros(m.n_dofs), f)[0]


LINEAR = {
    "pcg": dict(), "mixed": dict(method=1, inner_rtol=1e-2), "two_level": dict(coarse_nodes=200),
    "mixed_two_level": dict(method=1, inner_rtol=1e-2, coarse_nodes=200),
    "csr": dict(op="csr", op_outer="csr", rtol=1e-9), "csr_mixed": dict(op="csr", op_outer="csr", method=1, inner_rtol=1e-2, rtol=1e-9),
    "learned": dict(precond=1, learned_probe=8), "learned_two_level": dict(precond=1, learned_probe=8, coarse_nodes=200),
}


@pytest.mark.parametrize("polls", [None, 0, 2, 20])
@pytest.mark.parametrize("name", list(LINEAR))
def test_linear(direct, monkeypatch, name, polls):
    import jfem
    from jfem.learned import DEFAULT_WEIGHTS
    if polls is not None:
        monkeypatch.setenv("JFEM_PERSIST_POLLS", str(polls))
    m = box()
    kw = dict(dict(rtol=1e-10), **LINEAR[name])
    ctx = jfem.Context(0)
    ctx.upload(m)
    ctx.set_learned_weights(open(DEFAULT_WEIGHTS, "rb").read())
    say(f"resident waits: {name} polls={polls}")
    u = ctx.solve(**kw)[0]
    assert np.linalg.norm(u - direct) <= 100 * kw["rtol"] * np.linalg.norm(direct)
    solves, gave_up = ctx.resident_counts()
    say(f"{solves} resident solves, {gave_up} gave up")
    if polls is None:
        assert solves > 0 and gave_up == 0
    elif polls == 0:
        assert solves == 0 and gave_up == 1
    ctx.close()


@pytest.mark.parametrize("polls", [None, 0, 2, 20])
def test_heat_fit_and_newton(oracle, monkeypatch, polls):
    import jfem
    if polls is not None:
        monkeypatch.setenv("JFEM_PERSIST_POLLS", str(polls))
    m = box()
    rng = np.random.default_rng(3)
    k, q = np.exp(0.5 * rng.standard_normal(m.n_el)) * 3.0, rng.uniform(0.5, 2.0, m.n_el)
    nf = len(m.faces)
    flux, h, te = rng.uniform(0, 1, nf), rng.uniform(0.5, 1.0, nf), rng.uniform(10, 20, nf)
    fixed, Tf = np.isclose(m.X[:, 0], 0.0), np.full(m.n_nodes, 5.0)
    Kh, f = oracle.heat_system(m, k, q=q, faces=m.faces, ftype=m.ftype, flux=flux, h=h, T_ext=te)
    To = oracle.heat_solve_direct(Kh, f, fixed, Tf)
    u = rng.standard_normal(m.n_dofs) * 1e-3
    sig = oracle.lsq_fit(m, u, "stress")
    nl = M.box_tet10(19, 6, 3, seed=5, jitter=0.1, E_sigma=0.4, traction=(0.0, 0.0, -2.0))
    uo, _ = oracle.nh_newton(nl, load_steps=1, rtol=1e-10)

    def counted(call):
        ctx = jfem.Context(0)
        ctx.upload(nl)
        out = call(ctx)
        solves, gave_up = ctx.resident_counts()
        if polls is None:
            assert solves > 0 and gave_up == 0
        elif polls == 0:
            assert solves == 0 and gave_up > 0
        ctx.close()
        return out

    say(f"resident waits: heat polls={polls}")
    T = counted(lambda c: c.heat_solve(k, q, m.faces, flux=flux, h=h, T_ext=te, fixed=fixed, T_fixed=Tf, rtol=1e-12))[0]
    assert np.abs(T - To).max() <= 1e-8 * np.abs(To).max()
    say(f"resident waits: fits polls={polls}")
    out = counted(lambda c: c.postprocess(u))
    assert np.abs(out["stress_nodal"] - sig).max() <= 1e-9 * np.abs(sig).max()
    for method, coarse_nodes in ((0, 0), (1, 100)):
        say(f"resident waits: Newton polls={polls} method={method}")
        un = counted(lambda c: c.solve_nonlinear(load_steps=1, rtol=1e-10, method=method, coarse_nodes=coarse_nodes))[0]
        assert np.linalg.norm(un - uo) <= 1e-7 * np.linalg.norm(uo)


def cut(m, n_el):
    """The first n_el elements of m."""
    used, conn = np.unique(m.conn[:n_el], return_inverse=True)
    at = np.full(m.n_nodes, -1)
    at[used] = np.arange(len(used))
    clamp = at[m.clamp_nodes]
    return M.Mesh(X=m.X[used], conn=conn.reshape(n_el, -1), etype=m.etype, E=m.E[:n_el], nu=m.nu[:n_el], faces=np.zeros((0, 6), np.int64),
                  ftype="Tri6", clamp_nodes=clamp[clamp >= 0])


@pytest.mark.parametrize("n_el,resident", [(32768, True), (32769, False)])
def test_the_limit_of_the_element_kernels(n_el, resident):
    """256 patches of 128 Tet10 elements run resident, 257 do not.  Bar: the
    residual that the solve reports, with jfm_apply's product (another order of the
    sums: 1e-10 of the load)."""
    import jfem
    m = cut(M.box_tet10(18, 18, 17, L=(1.0, 1.0, 1.0), seed=5, jitter=0.1, E_sigma=0.4), n_el)
    f = np.random.default_rng(4).normal(size=m.n_dofs)
    free = ~m.fixed_mask().astype(bool).ravel()
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"limit of the element kernels: {n_el} elements")
    u, _, st = ctx.solve(f=f, rtol=1e-8)
    assert (ctx.resident_counts()[0] > 0) == resident and ctx.resident_counts()[1] == 0
    r = np.linalg.norm((f - ctx.apply(u))[free]) / np.linalg.norm(f[free])
    assert r <= 1e-8 + 1e-10 and abs(r - st["relres"]) <= 1e-10
    ctx.close()


def curved():
    m = box()
    X = m.X.copy()
    X[m.conn[0, 4]] += 0.01
    return M.Mesh(X=X, conn=m.conn, etype=m.etype, E=m.E, nu=m.nu, faces=m.faces, ftype=m.ftype, clamp_nodes=m.clamp_nodes,
                  traction=m.traction)


def orphan():
    m = box()
    return M.Mesh(X=np.vstack([m.X, m.X[:1] - 1.0]), conn=m.conn, etype=m.etype, E=m.E, nu=m.nu, faces=m.faces, ftype=m.ftype,
                  clamp_nodes=np.append(m.clamp_nodes, m.n_nodes), traction=m.traction)


@pytest.mark.parametrize("name,make,kw", [("curved", curved, dict()), ("orphan", orphan, dict()), ("ebe", box, dict(op="ebe")),
                                          ("csr_two_level", box, dict(op="csr", op_outer="csr", coarse_nodes=200)),
                                          ("coarse_too_large", box, dict(coarse_nodes=8))])
def test_launched_forms(oracle, name, make, kw):
    import jfem
    m = make()
    ud = oracle.solve_direct_lapack(oracle.assemble_csr(m), m.fixed_mask(), np.zeros(m.n_dofs), oracle.load_vector(m))[0]
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"launched: {name}")
    u = ctx.solve(rtol=1e-9, **kw)[0]
    assert np.linalg.norm(u - ud) <= 1e-7 * np.linalg.norm(ud)
    assert ctx.resident_counts() == (0, 0)
    ctx.close()


def test_resident_again_after_a_give_up(monkeypatch):
    """The call after a give-up, and every call on a new mesh, runs resident again,
    to the bits of a context that never gave up; while it happens again, one call,
    then one of two, then one of four tries."""
    import jfem
    m = box()
    kw = dict(rtol=1e-10)
    ctx = jfem.Context(0)
    ctx.upload(m)
    u = ctx.solve(**kw)[0]
    n = ctx.resident_counts()[0]
    monkeypatch.setenv("JFEM_PERSIST_POLLS", "0")
    say("resident again after a give-up")
    tried = []
    for _ in range(8):
        before = ctx.resident_counts()[1]
        ctx.solve(**kw)
        tried.append(ctx.resident_counts()[1] - before)
    assert tried == [1, 1, 0, 1, 0, 0, 0, 1]
    ctx.upload(m)
    ctx.solve(**kw)
    monkeypatch.delenv("JFEM_PERSIST_POLLS")
    assert ctx.resident_counts() == (n, 5)
    assert np.array_equal(ctx.solve(**kw)[0], u)
    assert ctx.resident_counts() == (2 * n, 5)
    ctx.close()


@pytest.mark.parametrize("patches", [(85, 85, 86), (80, 80, 80), (128, 128), (41, 43, 45, 47, 9)])
def test_solves_from_several_threads(patches):
    """Resident kernels of several contexts at once, workgroups that fill the device
    or more: none gives up, and each has the bits of its solves alone."""
    import jfem
    big = M.box_tet10(18, 18, 9, L=(2.0, 2.0, 1.0), seed=5, jitter=0.1, E_sigma=0.4)
    ms = [cut(big, 128 * n) for n in patches]
    f = [np.random.default_rng(4 + k).normal(size=m.n_dofs) for k, m in enumerate(ms)]
    cs = [jfem.Context(0) for _ in ms]
    kw = dict(rtol=1e-8, method=1, inner_rtol=1e-2)
    for c, m in zip(cs, ms):
        c.upload(m)
    alone = [c.solve(f=f[k], **kw)[0] for k, c in enumerate(cs)]
    say(f"resident solves side by side: {patches}")
    same = [[] for _ in cs]

    def work(k):
        for _ in range(6):
            same[k].append(np.array_equal(cs[k].solve(f=f[k], **kw)[0], alone[k]))

    th = [threading.Thread(target=work, args=(k,)) for k in range(len(cs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    counts = [c.resident_counts() for c in cs]
    say(f"solves, give-ups: {counts}")
    assert all(n > 0 and g == 0 for n, g in counts)
    assert all(s == [True] * 6 for s in same)
    for c in cs:
        c.close()


@pytest.mark.parametrize("gen,g,slots", [("box_tet10", (12, 12, 12), None), ("box_tet10", (30, 12, 12), None),
                                         ("box_hex8", (40, 40, 40), 61000)])
def test_long_elements(gen, g, slots):
    """Elements several times as long as wide (10 x 1 x 1): the resident form, whose
    patches do not fit until they are cut in element lengths, and for Hex8 compact
    480-element patches (the nodes' partial sums of the bounding box's scale within
    2%; one scale for all axes gave 133,534)."""
    import jfem
    m = getattr(M, gen)(*g, seed=1, jitter=0.1)
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"long elements: {gen} {g}")
    x = np.random.default_rng(2).normal(size=m.n_dofs)
    y, yc = ctx.apply(x), ctx.apply(x, op="csr")
    assert np.abs(y - yc).max() <= 1e-12 * np.abs(yc).max()
    if slots:
        assert ctx.info()["shared_slots"] <= slots
    kw = dict(rtol=1e-8, coarse_nodes=300)
    u = ctx.solve(**kw)[0]
    assert ctx.resident_counts()[0] > 0
    uc = ctx.solve(op="csr", op_outer="csr", **kw)[0]   # launched
    assert np.linalg.norm(u - uc) <= 1e-6 * np.linalg.norm(uc)
    ctx.close()


@pytest.mark.parametrize("gen,g,size,slots,resident", [
    ("box_hex8", (64, 32, 32), (10, 1, 1), 58000, True),      # 65,844 cut across the grid's halves
    ("box_hex8", (100, 25, 26), (1, 1, 1), 66000, False),     # 66,809
    ("box_tet10", (60, 20, 20), (10, 1, 1), 232000, False),   # 445,595 with one scale, 231,378 the bounding box's
    ("box_tet10", (26, 25, 24), (10, 1, 1), None, False)])
def test_patches_of_long_elements_along_the_grid(gen, g, size, slots, resident):
    """Element lengths count in whole halvings of the mesh's extent: patches as compact
    as those of the bounding box's scale, and resident where that fits."""
    import jfem
    m = getattr(M, gen)(*g, L=tuple(a * b / g[0] for a, b in zip(g, size)), seed=1, jitter=0.1)
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"long elements along the grid: {gen} {g}")
    x = np.random.default_rng(2).normal(size=m.n_dofs)
    yc = ctx.apply(x, op="csr")
    for y in (ctx.apply(x), ctx.apply(x, op="ebe")):
        assert np.abs(y - yc).max() <= 1e-12 * np.abs(yc).max()
    if slots:
        assert ctx.info()["shared_slots"] <= slots
    # 30 iterations (these meshes' conditioning leaves no residual of 1e-8 to some operators)
    kw = dict(rtol=1e-8, coarse_nodes=300, maxit=30, raise_on_noconv=False)
    u = ctx.solve(**kw)[0]
    assert (ctx.resident_counts()[0] > 0) == resident
    uc = ctx.solve(op="csr", op_outer="csr", **kw)[0]
    assert np.linalg.norm(u - uc) <= 1e-6 * np.linalg.norm(uc)
    ctx.close()
