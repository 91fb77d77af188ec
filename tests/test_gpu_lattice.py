"""Lattice levels smoothed in bricks (lattice_kernels.hpp, option lattice) against one launch per step
on the banded format (lattice = 0): the same row sums, steps and transfers in the same order, so cycles
are equal bit for bit.  The levels' sizes put the bricks' tiles at their edges: lattices smaller than a
tile, one node more than a multiple of it, and many tiles."""
import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch


def cycles(torch, H, d, inner, lattice, n=2, fmt="banded", **kw):
    from feat3_amd.solver import MGPCG
    s = MGPCG(H, inner=inner, fmt=fmt, options={"lattice": lattice, "tail_max_n": kw.pop("tail", 30)}, **kw).init()
    dd = torch.from_numpy(d).cuda()
    c = torch.empty_like(dd)
    for _ in range(n):      # a second cycle starts from the first one's buffers
        s.vcycle(c, dd)
    out, k = c.cpu().numpy(), s.info()["kernels_per_vcycle"]
    s.done()
    return out, k


def defect(H, seed=3):
    d = np.random.default_rng(seed).uniform(-1.0, 1.0, H.n)
    d[H.levels[0].bnd] = 0.0
    return d


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,deg,lvl", [(2, 1, 4), (2, 1, 6), (2, 1, 8), (2, 2, 4), (2, 2, 6), (3, 1, 3), (3, 1, 4), (3, 1, 5), (3, 1, 6)])
def test_bricks_are_bitwise_the_steps(torch, dim, deg, lvl, inner):
    H = pb.hierarchy(dim, deg, lvl, 1)
    d = defect(H)
    for cycle, pre, post in (("v", 4, 4), ("v", 1, 1), ("f", 2, 3), ("w", 3, 2)):
        if cycle == "w" and lvl > 5:
            continue
        a, ka = cycles(torch, H, d, inner, 1, cycle=cycle, pre=pre, post=post)
        b, kb = cycles(torch, H, d, inner, 0, cycle=cycle, pre=pre, post=post)
        assert ka < kb, (ka, kb)
        assert np.array_equal(a, b), (cycle, pre, post, np.abs(a - b).max())


@pytest.mark.parametrize("inner", ["f64", "f32"])
@pytest.mark.parametrize("lvl", [4, 7])
def test_variable_coefficient_bricks(torch, lvl, inner):
    """A row of values per node (no two alike)."""
    k = np.exp(np.random.default_rng(7).uniform(-1.0, 1.0, 1 << (2 * lvl)))
    H = pb.hierarchy(2, 1, lvl, 1, kcell=k)
    d = defect(H)
    a, ka = cycles(torch, H, d, inner, 1)
    b, kb = cycles(torch, H, d, inner, 0)
    assert ka < kb and np.array_equal(a, b)


@pytest.mark.parametrize("dim,deg,lvl", [(2, 1, 6), (2, 2, 5), (3, 1, 4)])
def test_changed_rows_are_not_taken_as_uniform(torch, dim, deg, lvl):
    """One inner row with another diagonal, and Dirichlet nodes besides the boundary: 3D and Q2 levels keep
    their steps (one kernel each), 2D Q1 levels take rows of their own; the cycles stay equal."""
    H = pb.hierarchy(dim, deg, lvl, 1)
    A = H.levels[0].A
    rows = np.repeat(np.arange(A.rows), np.diff(A.row_ptr.astype(np.int64)))
    mid = A.rows // 2
    A.val[(A.col_ind == rows) & (rows == mid)] *= 1.5
    d = defect(H)
    a, ka = cycles(torch, H, d, "f64", 1)
    b, kb = cycles(torch, H, d, "f64", 0)
    assert np.array_equal(a, b)
    G = pb.hierarchy(dim, deg, lvl, 1)
    G.levels[0].bnd = np.union1d(G.levels[0].bnd, np.array([mid + 1], np.uint32)).astype(np.uint32)
    d = defect(G)
    a, ka = cycles(torch, G, d, "f32", 1)
    b, kb = cycles(torch, G, d, "f32", 0)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("inner", ["f64", "f32"])
@pytest.mark.parametrize("dim,deg,lvl", [(2, 1, 6), (2, 2, 5), (3, 1, 4)])
@pytest.mark.parametrize("where", ["all", "one"])
def test_two_entries_of_one_column_are_added(torch, dim, deg, lvl, inner, where):
    """An entry stored as two halves (exact) of one column, in every inner row or in one: the general formats
    add them, so such a level is no lattice.  The cycles agree with the whole entry's to the rounding of a
    row sum (25 or 27 terms); with bands on the other levels they are those of lattice = 0 bit for bit."""
    H = pb.hierarchy(dim, deg, lvl, 1)
    A = H.levels[0].A
    rows = np.repeat(np.arange(A.rows), np.diff(A.row_ptr.astype(np.int64)))
    inner_row = np.ones(A.rows, bool)
    inner_row[H.levels[0].bnd] = False
    pick = np.flatnonzero((A.col_ind == rows + 1) & inner_row[rows] & inner_row[np.minimum(rows + 1, A.rows - 1)])
    if where == "one":
        pick = pick[pick.size // 2:][:1]
    d = defect(H)
    whole, _ = cycles(torch, H, d, inner, 0, fmt="csr")
    times = np.ones(A.nnz, np.int64)
    times[pick] = 2
    ends = np.cumsum(times)
    val = np.repeat(A.val, times)
    val[ends[pick] - 1] *= 0.5
    val[ends[pick] - 2] *= 0.5
    rp = np.concatenate([[0], ends])[A.row_ptr.astype(np.int64)].astype(np.uint32)
    H.levels[0].A = pb.Csr(A.rows, A.cols, rp, np.repeat(A.col_ind, times), val)
    eps = np.finfo(np.float64 if inner == "f64" else np.float32).eps
    for fmt in ("csr", "banded"):
        a, _ = cycles(torch, H, d, inner, 1, fmt=fmt)
        b, _ = cycles(torch, H, d, inner, 0, fmt=fmt)
        assert fmt == "csr" or np.array_equal(a, b), np.abs(a - b).max()
        assert np.linalg.norm(a - whole) <= 27 * eps * np.linalg.norm(whole)


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,deg,lvl,coef", [(2, 1, 7, False), (2, 1, 7, True), (2, 2, 6, False), (3, 1, 5, False)])
def test_dirichlet_rows_that_are_not_finite(torch, dim, deg, lvl, coef, inner):
    """A NaN or an infinity in the matrix row of a Dirichlet node of the finest or the next level: the cycle
    carries it and the solve ends with status aborted, as with the row kernels (lattice = 0)."""
    from feat3_amd.solver import MGPCG
    k = np.exp(np.random.default_rng(7).uniform(-1.0, 1.0, 1 << (2 * lvl))) if coef else None
    for level, bad in ((0, np.nan), (0, np.inf), (1, np.nan)):
        H = pb.hierarchy(dim, deg, lvl, 1, kcell=k)
        L = H.levels[level]
        L.A.val[int(L.A.row_ptr[int(L.bnd[L.bnd.size // 3])])] = bad
        b = torch.from_numpy(pb.filtered_rhs(H, 0)).cuda()
        out = []
        for lattice in (1, 0):
            s = MGPCG(H, inner=inner, options={"lattice": lattice}).init()
            out.append(s.correct(torch.zeros_like(b), b))
            s.done()
        assert out[0] == out[1] and out[0][0] == 3, (level, bad, out)


@pytest.mark.parametrize("fmt", ["csr", "sell"])
@pytest.mark.parametrize("inner", ["f64", "f32"])
def test_other_formats_agree(torch, fmt, inner):
    """The general formats round their products before adding them, the bricks do not: a row sum of w = 27
    terms differs by at most w eps of its absolute terms, the cycle by a few times that."""
    H = pb.hierarchy(3, 1, 4, 1)
    d = defect(H)
    a, _ = cycles(torch, H, d, inner, 1, fmt=fmt)
    b, _ = cycles(torch, H, d, inner, 0, fmt=fmt)
    eps = np.finfo(np.float64 if inner == "f64" else np.float32).eps
    assert np.linalg.norm(a - b) <= 27 * eps * np.linalg.norm(b)


@pytest.mark.parametrize("inner", ["f64", "f32"])
def test_columns_are_bitwise_the_steps(torch, inner):
    """The finest 3D level of 2^20 rows or more takes its steps by columns (129^3 nodes): the cycle bit for
    bit; the solve, whose dot products are grouped by other blocks, the same iterations and 1e-12."""
    from feat3_amd.solver import MGPCG
    levels = pb.hierarchy_device(3, 1, 7, 1)
    n = levels[0].A.rows
    b = torch.rand(n, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(3)) - 0.5
    b[levels[0].bnd.long()] = 0.0
    out = []
    for lattice in (1, 0):
        s = MGPCG(levels, inner=inner, fmt="banded", options={"lattice": lattice}).init()
        info = s.info()
        assert (info["column_levels"], info["outer_columns"]) == (lattice, lattice)
        c = torch.empty_like(b)
        for _ in range(2):
            s.vcycle(c, b)
        x = torch.zeros_like(b)
        st, it = s.correct(x, b)
        # from a start other than zero: the initial defect's product
        y = 0.5 * x
        st2, it2 = s.correct(y, b)
        out.append((c.cpu().numpy(), x.cpu().numpy(), y.cpu().numpy(), st, it, st2, it2))
        s.done()
    a, e = out
    assert np.array_equal(a[0], e[0])
    assert a[3:] == e[3:] and a[3] == a[5] == 2
    assert np.linalg.norm(a[1] - e[1]) <= 1e-12 * np.linalg.norm(e[1])
    assert np.linalg.norm(a[2] - e[2]) <= 1e-12 * np.linalg.norm(e[2])


@pytest.mark.parametrize("dim,deg,lvl", [(2, 1, 6), (2, 2, 5), (3, 1, 5)])
@pytest.mark.parametrize("inner", ["f64", "f32"])
def test_row_kernels_with_and_without_tensor_transfers(torch_cuda, dim, deg, lvl, inner):
    """Without the lattice kernels (lattice = 0) the tensor transfers and the stored ones give the same
    solve bit for bit; with them the option changes nothing either."""
    from feat3_amd.solver import MGPCG
    torch = torch_cuda
    print(f"case transfers {dim}D Q{deg} L{lvl} {inner}", flush=True)
    H = pb.hierarchy(dim, deg, lvl, 1)
    b = torch.from_numpy(pb.filtered_rhs(H, 0)).cuda()
    for lattice in (0, 1):
        out = []
        for tensor in (1, 0):
            s = MGPCG(H, inner=inner, fmt="banded", options={"lattice": lattice, "tensor_transfer": tensor}).init()
            x = torch.zeros_like(b)
            st, it = s.correct(x, b)
            out.append((st, it, x.cpu().numpy()))
            s.done()
        assert out[0][:2] == out[1][:2] and np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("dim,deg,lvl,coef,route", [(2, 1, 7, False, 1), (2, 1, 7, True, 1), (2, 2, 6, False, 1), (3, 1, 5, False, 1),
                                                    (3, 1, 7, False, 2), (3, 2, 3, False, 0)])
def test_info_tells_the_route_and_its_bytes(torch, dim, deg, lvl, coef, route):
    """info() names the way the finest level is smoothed; the cycle's bytes are those of its launches: on
    lattice levels vectors only (at most five of the level and three of the next one a launch; ten more
    with a row of values per node), so fewer than with one launch per step."""
    from feat3_amd.solver import MGPCG
    k = torch.exp(torch.rand(1 << (2 * lvl), dtype=torch.float64, device="cuda")) if coef else None
    levels = pb.hierarchy(dim, deg, lvl, 1) if deg == 2 and dim == 3 else pb.hierarchy_device(dim, deg, lvl, 1, k)
    info = []
    for lattice in (1, 0):
        s = MGPCG(levels, inner="f32", options={"lattice": lattice}).init()
        info.append(s.info())
        s.done()
    a, b = info
    upper = a["levels"] - a["tail_levels"]
    assert a["finest_lattice"] == route and b["finest_lattice"] == 0
    assert (a["brick_levels"], a["column_levels"]) == {0: (0, 0), 1: (upper, 0), 2: (upper - 1, 1)}[route]
    assert b["brick_levels"] == b["column_levels"] == b["outer_columns"] == 0 and a["outer_columns"] == (route == 2)
    assert a["tail_matrices"] == b["tail_matrices"] == 1
    assert (a["vcycle_bytes"] < b["vcycle_bytes"]) == (route > 0) and (a["outer_bytes"] < b["outer_bytes"]) == (route > 0)
    if route == 1:
        m = ((deg << lvl) + 1) ** dim
        tail = 2 * 4 * 1100 + 8 * 1100 ** 2
        assert a["vcycle_bytes"] <= a["kernels_per_vcycle"] * 4 * m * (8 + (10 if coef else 0)) + tail


@pytest.mark.parametrize("inner,fmt,cycle,pre,post", [
    ("f32", "banded", "v", 1, 3),      # the entry writes the first iterate and the defect follows it
    ("f64", "banded", "v", 2, 2),      # the step that forms the entry's iterate, then the defect
    ("f32", "banded", "f", 3, 1),      # the cycle's last step is the only one behind the prolongation
    ("f16", "banded", "v", 4, 4), ("f16", "banded", "f", 1, 1), ("f64", "banded", "f", 4, 4),
    ("f32", "csr", "v", 4, 4), ("f16", "sell", "v", 2, 3)])
def test_columns_in_every_cycle(torch, inner, fmt, cycle, pre, post):
    """129^3 nodes by columns against one launch per step: the cycle bit for bit with bands (rounding of the
    products in the general formats, as test_other_formats_agree), the solve's iterations alike."""
    from feat3_amd.solver import MGPCG
    print(f"case columns {inner} {fmt} {cycle}({pre},{post})", flush=True)
    levels = pb.hierarchy_device(3, 1, 7, 1)
    n = levels[0].A.rows
    b = torch.rand(n, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(3)) - 0.5
    b[levels[0].bnd.long()] = 0.0
    out = []
    for lattice in (1, 0):
        s = MGPCG(levels, inner=inner, fmt=fmt, cycle=cycle, pre=pre, post=post, options={"lattice": lattice}).init()
        assert (s.info()["column_levels"], s.info()["outer_columns"]) == (lattice, lattice)
        c, x = torch.empty_like(b), torch.zeros_like(b)
        for _ in range(2):
            s.vcycle(c, b)
        r = s.correct(x, b)
        out.append((c, x, r))
        s.done()
    (c, x, r), (d, y, q) = out
    eps = 2.0 ** -52 if inner == "f64" else 2.0 ** -23
    if fmt == "banded":
        assert torch.equal(c, d)
    else:
        assert float((c - d).norm()) <= 27 * eps * float(d.norm())
    assert r == q and r[0] == 2
    # FP64 dot products of 2e6 terms grouped by other blocks; other formats: cycles that differ by rounding
    assert float((x - y).norm()) <= (1e-12 if fmt == "banded" else 1e-8) * float(y.norm())


@pytest.mark.parametrize("dim,lvl,inner", [(2, 11, "f32"), (3, 8, "f32"), (3, 8, "f64")])
def test_sums_of_more_blocks_than_are_folded(torch, dim, lvl, inner):
    """The cycle's last launch and, in 3D, the outer product leave more partial sums than every block of
    the next kernel adds up (2048): a launch of its own adds them.  2049^2 nodes: 3182 blocks; 257^3
    nodes: 8385 (FP32) and 8450.  Against one launch per step: the same iterations.  The dot products are
    grouped otherwise (2e7 terms, 1e-16 each), so the defects differ in their last digits, and a value
    of them may round to the other FP32 neighbour for the cycle: that changes a correction by at most
    u = 6e-8 of its norm, the next defect by as much of the one before, and the solution by as much."""
    from feat3_amd.solver import MGPCG
    print(f"case many partials {dim}D L{lvl} {inner}", flush=True)
    levels = pb.hierarchy_device(dim, 1, lvl, 1)
    n = levels[0].A.rows
    b = torch.rand(n, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(5)) - 0.5
    b[levels[0].bnd.long()] = 0.0
    out = []
    for lattice in (1, 0):
        s = MGPCG(levels, inner=inner, fmt="banded", options={"lattice": lattice}).init()
        assert s.info()["finest_lattice"] == lattice * (dim - 1) and s.info()["outer_columns"] == lattice * (dim - 2)
        x = torch.zeros_like(b)
        out.append((s.correct(x, b), x, s.history()))
        s.done()
    (r, x, h), (q, y, g) = out
    assert r == q and r[0] == 2
    assert h[0] == pytest.approx(g[0], rel=1e-12)
    assert (np.abs(h - g)[1:] <= 2.0 ** -24 * g[:-1]).all(), (h, g)
    assert float((x - y).norm()) <= 2.0 ** -24 * float(y.norm())


def lattice_hierarchy(dim, deg, cells):
    """Laplacians of 2^k * c cells per axis with the two-level transfers, coarsened while the cells are even."""
    import scipy.sparse as sp
    H = pb.Hierarchy(dim, deg)

    def csr(M):
        M = sp.csr_matrix(M)
        M.sort_indices()
        return pb.Csr(M.shape[0], M.shape[1], M.indptr.astype(np.uint32), M.indices.astype(np.uint32), M.data.astype(np.float64))

    def line(c):
        k = np.array([[1, -1], [-1, 1]]) if deg == 1 else np.array([[7, -8, 1], [-8, 16, -8], [1, -8, 7]]) / 3.0
        w = np.array([[2, 1], [1, 2]]) / 6.0 if deg == 1 else np.array([[4, 2, -1], [2, 16, 2], [-1, 2, 4]]) / 30.0
        K, M = np.zeros((deg * c + 1,) * 2), np.zeros((deg * c + 1,) * 2)
        for e in range(c):
            i = slice(deg * e, deg * e + deg + 1)
            K[i, i] += k
            M[i, i] += w
        return sp.csr_matrix(K), sp.csr_matrix(M)

    def prol(c):
        m = deg * c + 1
        P = np.zeros((m, deg * c // 2 + 1))
        for i in range(m):
            if deg == 1:
                P[i, i // 2] += 0.5
                P[i, (i + 1) // 2] += 0.5
            else:
                e, t = min(i // 4, c // 2 - 1), (i - 4 * min(i // 4, c // 2 - 1)) / 4.0
                P[i, 2 * e:2 * e + 3] = [(1 - t) * (1 - 2 * t), 4 * t * (1 - t), t * (2 * t - 1)]
        return sp.csr_matrix(P)

    def kron(fs):
        out = fs[0]
        for f in fs[1:]:
            out = sp.kron(f, out, format="csr")
        return out
    while True:
        K, M = line(cells)
        A = sum(kron([K if a == ax else M for a in range(dim)]) for ax in range(dim))
        m = deg * cells + 1
        edge = np.zeros((m,) * dim, bool)
        for ax in range(dim):
            edge[(slice(None),) * ax + (0,)] = edge[(slice(None),) * ax + (-1,)] = True
        L = pb.Level(csr(A), np.flatnonzero(edge.ravel()).astype(np.uint32))
        H.levels.append(L)
        if cells % 2 or m ** dim <= 130:
            return H
        P = kron([prol(cells)] * dim)
        L.P, L.R = csr(P), csr(P.T)
        cells //= 2


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,deg,cells", [(2, 1, 20), (2, 1, 44), (2, 1, 104), (2, 2, 12), (2, 2, 20), (2, 2, 44), (3, 1, 10),
                                           (3, 1, 12), (3, 1, 20), (3, 1, 36)])
def test_lattices_of_other_sizes(torch, dim, deg, cells, inner):
    """Lattices whose cells per axis are no power of two (and coarse ones with an even number of nodes)."""
    H = lattice_hierarchy(dim, deg, cells)
    d = defect(H)
    for cycle, pre, post in (("v", 4, 4), ("f", 1, 2)):
        a, ka = cycles(torch, H, d, inner, 1, cycle=cycle, pre=pre, post=post)
        b, kb = cycles(torch, H, d, inner, 0, cycle=cycle, pre=pre, post=post)
        assert ka < kb, (ka, kb)
        assert np.array_equal(a, b), (cycle, pre, post, np.abs(a - b).max())
