"""The lists that an upload builds on the device (mesh_lists.hip), through the C ABI.

A star of tetrahedra around one node: its row of the pattern has thousands of
contributions (more than the LDS of the row kernel holds: 1,024), beside rows of
a few.  One element, nodes in random order, and nodes of no element.  The
pattern is compared exactly with the one of the elements, the values with the
oracle's assembly (1e-13 of the largest: the same FP64 sums, in element order),
and a solve on the star, one of whose nodes lies in every patch, with the
oracle's direct solve (rtol 1e-10: 1e-8, as the resident PCG's tests ask).
"""
import numpy as np
import pytest

from jfem import mesh as M

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu] {msg}", flush=True)


def star(n, quadratic):
    """The tetrahedra between the centre of a cube and its surface of 12 n^2 triangles."""
    b = M.box_tet4(n, n, n, L=(1.0, 1.0, 1.0))
    f = np.concatenate([b.conn[:, list(c)] for c in ((0, 2, 1), (0, 1, 3), (1, 2, 3), (0, 3, 2))])
    _, first, count = np.unique(np.sort(f, 1), axis=0, return_index=True, return_counts=True)
    tri = f[first[count == 1]]
    used, tri = np.unique(tri, return_inverse=True)
    tri = tri.reshape(-1, 3)
    X = np.vstack([b.X[used], [[0.5, 0.5, 0.5]]])
    conn = np.column_stack([tri[:, 0], tri[:, 2], tri[:, 1], np.full(len(tri), len(used))])
    if quadratic:
        e = np.sort(conn[:, [[0, 1], [1, 2], [2, 0], [0, 3], [1, 3], [2, 3]]], 2)
        ed, mid = np.unique(e.reshape(-1, 2), axis=0, return_inverse=True)
        X, conn = np.vstack([X, 0.5 * (X[ed[:, 0]] + X[ed[:, 1]])]), np.column_stack([conn, len(X) + mid.reshape(-1, 6)])
    E = np.exp(np.random.default_rng(1).normal(0.0, 0.4, len(conn)))
    return M.Mesh(X=X, conn=conn, etype="Tet10" if quadratic else "Tet4", E=E, nu=np.full(len(conn), 0.3),
                  faces=np.zeros((0, 3), np.int64), ftype="Tri3", clamp_nodes=np.flatnonzero(X[:, 0] == 0.0))


def shuffled(m, extra):
    """Nodes in random order, `extra` of them in no element."""
    rng = np.random.default_rng(2)
    N = m.n_nodes + extra
    new = rng.permutation(N)[:m.n_nodes]
    X = rng.uniform(0.0, 1.0, (N, 3))
    X[new] = m.X
    return M.Mesh(X=X, conn=new[m.conn], etype=m.etype, E=m.E, nu=m.nu, faces=np.zeros((0, 3), np.int64), ftype="Tri3",
                  clamp_nodes=new[m.clamp_nodes])


def one_hex():
    m = M.box_hex8(1, 1, 1)
    return M.Mesh(X=m.X, conn=m.conn, etype="Hex8", E=m.E, nu=m.nu, faces=np.zeros((0, 4), np.int64), ftype="Quad4",
                  clamp_nodes=m.clamp_nodes)


CASES = {
    "one_hex8": one_hex,
    "star_tet4": lambda: star(9, False),      # 972 elements: 3,888 entries
    "star_tet10": lambda: star(4, True),      # 192 elements: 1,920 entries
    "star_tet10_at_the_limit": lambda: star(3, True),  # 108: 1,080
    "shuffled_hex8": lambda: shuffled(M.box_hex8(5, 4, 3, jitter=0.1, seed=3), 0),
    "shuffled_tet10_orphans": lambda: shuffled(M.box_tet10(5, 4, 3, jitter=0.1, seed=3), 7),
}


@pytest.mark.parametrize("name", list(CASES))
def test_pattern_and_values(oracle, name):
    import jfem
    m = CASES[name]()
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"mesh lists {name}: nodes={m.n_nodes} el={m.n_el}")
    rp, ci = ctx.csr_pattern()
    rows = [[] for _ in range(m.n_nodes)]
    for c in m.conn:
        for a in c:
            rows[a].append(c)
    ptr, col = [0], []
    for r in rows:
        dofs = (3 * np.unique(np.concatenate(r))[:, None] + np.arange(3)).ravel() if r else np.zeros(0, np.int64)
        for _ in range(3):
            col.append(dofs)
            ptr.append(ptr[-1] + len(dofs))
    assert np.array_equal(rp, ptr) and np.array_equal(ci, np.concatenate(col))
    vals = ctx.assemble()
    vals = vals[0] if isinstance(vals, tuple) else vals
    import scipy.sparse as sp
    ro, co, vo = oracle.assemble_csr(m)
    Ko = sp.csr_matrix((vo, co, ro), shape=(m.n_dofs, m.n_dofs))
    K = sp.csr_matrix((vals, ci, rp), shape=(m.n_dofs, m.n_dofs))
    assert abs(K - Ko).max() <= 1e-13 * np.abs(vo).max()
    ctx.close()


@pytest.mark.parametrize("name", ["star_tet4", "star_tet10"])
def test_solve_on_a_star(oracle, name):
    import jfem
    m = CASES[name]()
    f = np.random.default_rng(4).normal(size=m.n_dofs)
    ud, _, _ = oracle.solve_direct_lapack(oracle.assemble_csr(m), m.fixed_mask(), np.zeros(m.n_dofs), f)
    ctx = jfem.Context(0)
    ctx.upload(m)
    for kw in (dict(method=0), dict(method=1, inner_rtol=1e-2), dict(method=1, inner_rtol=1e-2, coarse_nodes=60)):
        say(f"solve {name} {kw}")
        u, _, _ = ctx.solve(f=f, rtol=1e-10, **kw)
        assert np.linalg.norm(u - ud) <= 1e-8 * np.linalg.norm(ud)
    ctx.close()


def fan(n, quadratic):
    """The tetrahedra between a point and 2 n^2 triangles of a square below it."""
    x = np.linspace(-1.0, 1.0, n + 1)
    X, Y = np.meshgrid(x, x, indexing="ij")
    i, j = (a.ravel() for a in np.meshgrid(np.arange(n), np.arange(n), indexing="ij"))
    at = lambda a, b: a * (n + 1) + b
    tri = np.concatenate([np.column_stack([at(i, j), at(i + 1, j), at(i, j + 1)]),
                          np.column_stack([at(i + 1, j), at(i + 1, j + 1), at(i, j + 1)])])
    X = np.vstack([np.column_stack([X.ravel(), Y.ravel(), np.zeros(X.size)]), [[0.1, 0.2, 1.0]]])
    conn = np.column_stack([tri, np.full(len(tri), len(X) - 1)])
    conn = conn[np.random.default_rng(1).permutation(len(conn))]
    if quadratic:
        e = np.sort(conn[:, [[0, 1], [1, 2], [2, 0], [0, 3], [1, 3], [2, 3]]], 2)
        ed, mid = np.unique(e.reshape(-1, 2), axis=0, return_inverse=True)
        X, conn = np.vstack([X, 0.5 * (X[ed[:, 0]] + X[ed[:, 1]])]), np.column_stack([conn, len(X) + mid.reshape(-1, 6)])
    return M.Mesh(X=X, conn=conn, etype="Tet10" if quadratic else "Tet4", E=np.full(len(conn), 1e3), nu=np.full(len(conn), 0.3),
                  faces=np.zeros((0, 3), np.int64), ftype="Tri3", clamp_nodes=np.flatnonzero((X[:, 2] == 0.0) & (X[:, :2].min(1) == -1.0)))


# entries of the largest row: 39,200 (ten sorted runs), 18,000, 8,192 (two full runs), 2,592
@pytest.mark.parametrize("n,quadratic", [(70, False), (30, True), (32, False), (18, False)])
def test_large_rows(oracle, n, quadratic):
    """Rows of nodes with thousands of elements: the pattern and the values, and an
    upload (once the device is warm) that takes less than 0.1 s (comparing all
    pairs of entries took 0.14 s at 1,922 Tet4 around a node, 0.3 s at 968 Tet10,
    sixteen times as long at four times as many)."""
    import time

    import scipy.sparse as sp
    import jfem
    m = fan(n, quadratic)
    ctx = jfem.Context(0)
    say(f"large rows: {m.n_el} {m.etype} around a node")
    ctx.upload(M.box_tet10(2, 2, 2))
    ctx.upload(fan(4, quadratic))
    t = time.perf_counter()
    ctx.upload(m)
    t = time.perf_counter() - t
    say(f"upload {1e3 * t:.1f} ms")
    rp, ci = ctx.csr_pattern()
    vals = ctx.assemble()[0]
    ro, co, vo = oracle.assemble_csr(m)
    assert np.array_equal(rp, ro) and np.array_equal(ci, co)
    assert np.abs(vals - vo).max() <= 1e-13 * np.abs(vo).max()
    assert t <= 0.1
    ctx.close()


# patches of the launched and of the resident form: 21 and 20; 4 and 15; 34 and 32 (one more
# than the resident form's lists hold)
@pytest.mark.parametrize("n,quadratic,resident", [(70, False, True), (30, True, True), (90, False, False)])
def test_patches_around_a_node(oracle, n, quadratic, resident):
    """A node that lies in every patch: products of the patch operator against the
    oracle's matrix (1e-12, the bar of jfm_apply), a resident solve against the
    launched assembled one (100 times rtol), and the time to make the patches (below
    the 40 ms that a quarter of these elements took one thread)."""
    import time

    import jfem
    m = fan(n, quadratic)
    x = np.random.default_rng(4).normal(size=m.n_dofs)
    csr = oracle.assemble_csr(m)
    ref = oracle.spmv(csr, x) * (1 - m.fixed_mask().ravel())
    ctx = jfem.Context(0)
    ctx.upload(fan(4, quadratic))
    ctx.apply(np.ones(3 * fan(4, quadratic).n_nodes))
    ctx.upload(m)
    say(f"patches around a node: {m.n_el} {m.etype}")
    t = time.perf_counter()
    y = ctx.apply(x)
    t = time.perf_counter() - t
    say(f"first product {1e3 * t:.1f} ms, {ctx.info()['n_patches']} patches")
    assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
    assert np.array_equal(y, ctx.apply(x))
    assert t <= 0.03
    f = np.random.default_rng(5).normal(size=m.n_dofs)
    ud = ctx.solve(f=f, op="csr", op_outer="csr", coarse_nodes=100, rtol=1e-9)[0]
    assert ctx.resident_counts() == (0, 0)
    t = time.perf_counter()
    u = ctx.solve(f=f, rtol=1e-9)[0]
    say(f"first solve {1e3 * (time.perf_counter() - t):.1f} ms, resident: {ctx.resident_counts()[0]}")
    assert (ctx.resident_counts()[0] > 0) == resident
    assert np.linalg.norm(u - ud) <= 1e-7 * np.linalg.norm(ud)
    ctx.close()


@pytest.mark.parametrize("n,quadratic", [(4, False), (6, False), (15, False), (6, True), (22, True)])
def test_iterations_around_a_node(n, quadratic):
    """A node of 32 to 968 elements in the resident form, whose sums the wave then
    forms together: the launched assembled solve's answer (100 times rtol), the same
    bits again, and below 15 us an iteration (the node's lane alone: 50 with 450 Tet4
    in a patch; launched 33)."""
    import jfem
    m = fan(n, quadratic)
    f = np.random.default_rng(5).normal(size=m.n_dofs)
    ctx = jfem.Context(0)
    ctx.upload(m)
    say(f"iterations around a node: {m.n_el} {m.etype}")
    ud = ctx.solve(f=f, op="csr", op_outer="csr", coarse_nodes=100, rtol=1e-10)[0]
    for kw in (dict(), dict(method=1, inner_rtol=1e-2), dict(coarse_nodes=60)):
        u = ctx.solve(f=f, rtol=1e-10, **kw)[0]
        u2, _, st = ctx.solve(f=f, rtol=1e-10, **kw)
        assert np.linalg.norm(u - ud) <= 1e-8 * np.linalg.norm(ud)
        assert np.array_equal(u, u2)
        if not kw:
            say(f"{1e3 * st['solve_ms'] / st['iterations']:.1f} us an iteration")
            assert st["solve_ms"] <= 0.2 + 0.015 * st["iterations"]
    assert ctx.resident_counts()[0] > 0
    ctx.close()
