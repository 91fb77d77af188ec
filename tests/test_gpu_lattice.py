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
