"""The coarse tail of the multigrid cycle applied as one matrix product per segment (mgpcg.hip,
build_tail_mats) against the same steps launched level by level (option tail_max_n = 0).

Bars: both evaluate the same linear map; a smoothing step, transfer or matrix product of a row of w
terms rounds with at most (w + 3) eps relative to its absolute terms, and the tail has at most about 50
dependent steps, whose errors the smoothers damp.  FP64 1e-12, FP32 and binary16 values 64 eps = 7.6e-6
(2-norm, relative); measured 2e-15 and 2e-7."""
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


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,deg,lvl,cycle", [(2, 1, 2, "v"), (2, 1, 5, "v"), (2, 1, 6, "f"), (2, 1, 6, "w"), (2, 2, 5, "v"),
                                               (3, 1, 2, "v"), (3, 1, 4, "f"), (3, 1, 4, "w"), (3, 2, 2, "v")])
def test_tail_matrix_matches_the_steps(torch, dim, deg, lvl, cycle, inner):
    from feat3_amd.solver import MGPCG
    H = pb.hierarchy(dim, deg, lvl, 1)
    d = np.random.default_rng(5).uniform(-1.0, 1.0, H.n)
    d[H.levels[0].bnd] = 0.0
    dd = torch.from_numpy(d).cuda()
    out = []
    for tail in (1100, 0):
        s = MGPCG(H, inner=inner, cycle=cycle, options={"tail_max_n": tail}).init()
        assert (s.info()["tail_levels"] > 0) == (tail > 0 and lvl > 1)
        assert (s.info()["tail_matrices"] > 0) == (tail > 0 and lvl > 1)
        c = torch.empty_like(dd)
        for _ in range(2):      # a second cycle starts from the first one's buffers
            s.vcycle(c, dd)
        out.append(c.cpu().numpy())
        s.done()
    err = np.linalg.norm(out[0] - out[1]) / np.linalg.norm(out[1])
    print(f"  {dim}D Q{deg} level {lvl} {cycle} {inner}: {err:.2e}", flush=True)
    assert err <= (1e-12 if inner == "f64" else 64 * np.finfo(np.float32).eps)


def exact_cycle(H, d, L=0):
    """The V(4,4) cycle in extended precision (np.longdouble), sparse matrices as they are."""
    T = np.longdouble

    def mul(M, v):
        out = np.zeros(M.rows, T)
        rows = np.repeat(np.arange(M.rows), np.diff(M.row_ptr.astype(np.int64)))
        np.add.at(out, rows, M.val.astype(T) * v[M.col_ind.astype(np.int64)])
        return out
    A, bnd = H.levels[L].A, H.levels[L].bnd
    rows = np.repeat(np.arange(A.rows), np.diff(A.row_ptr.astype(np.int64)))
    diag = A.val[A.col_ind == rows].astype(T)
    dinv = T(0.5) / diag
    dinv[bnd] = 0
    if H.levels[L].P is None:      # one inner node
        return d * dinv * 2
    x = dinv * d
    for _ in range(3):
        x = x + dinv * (d - mul(A, x))
    r = d - mul(A, x)
    r[bnd] = 0
    r = mul(H.levels[L].R, r)
    r[H.levels[L + 1].bnd] = 0
    c = mul(H.levels[L].P, exact_cycle(H, r, L + 1))
    c[bnd] = 0
    x = x + c
    for _ in range(4):
        x = x + dinv * (d - mul(A, x))
    return x


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,lvl", [(2, 2), (2, 4), (2, 5), (3, 2), (3, 3)])
def test_tail_matrix_rounds_once(torch, dim, lvl, inner):
    """Oscillatory, random and smooth right-hand sides, whose cycle on the tail is up to 100 times smaller
    than |M| |b|: the product is that of the exact linear map, rounded once per value, so its relative
    error (2-norm) is at most the unit roundoff u of the cycle's arithmetic.  The matrices are scaled to
    whole numbers (2D 8 and -1, 3D 32, 0, -2 and -1), which every storage holds exactly, as it does dinv
    and the coarse inverse.  Matrices of the cycle's own precision: up to 22 u."""
    from feat3_amd.solver import MGPCG
    H = pb.hierarchy(dim, 1, lvl, 1)
    for i, L in enumerate(H.levels):
        L.A.val = np.rint(L.A.val * (3.0 if dim == 2 else 12.0 * 2 ** (lvl - i)))
    m = 2 ** lvl + 1
    g = np.indices([m] * dim)
    cases = {"checkerboard": np.where(g.sum(0) % 2 == 0, 1.0, -1.0).ravel(), "lines": np.where(g[-1] % 2 == 0, 1.0, -1.0).ravel(),
             "random": np.random.default_rng(5).integers(-1000, 1000, m ** dim).astype(np.float64),
             "smooth": np.rint(1000 * np.prod(np.sin(np.pi * g / (m - 1)), axis=0)).ravel()}
    s = MGPCG(H, inner=inner).init()
    assert s.info()["tail_levels"] == lvl
    u = 2.0 ** -53 if inner == "f64" else 2.0 ** -24
    for name, d in cases.items():
        d[H.levels[0].bnd] = 0.0
        c = torch.empty(m ** dim, dtype=torch.float64, device="cuda")
        s.vcycle(c, torch.from_numpy(d).cuda())
        e = exact_cycle(H, d.astype(np.longdouble))
        err = float(np.linalg.norm((c.cpu().numpy() - e).astype(np.float64)) / np.linalg.norm(e.astype(np.float64)))
        print(f"  {dim}D level {lvl} {inner} {name}: {err / u:.3f} u", flush=True)
        assert err <= 1.001 * u
    s.done()


@pytest.mark.parametrize("dim,deg,lvl,cycle,coef", [(2, 1, 5, "v", False), (2, 1, 5, "f", False), (2, 1, 4, "w", True), (2, 2, 4, "v", False),
                                                    (3, 1, 3, "v", False), (2, 1, 5, "v", True)])
def test_fp32_tail_does_not_carry_the_rounded_values(torch, dim, deg, lvl, cycle, coef):
    """The matrix of an FP32 cycle's tail is formed from the FP64 level matrices: with a right-hand side that
    FP32 holds, the result is the FP64 cycle's rounded once (at most the unit roundoff, 2-norm)."""
    from feat3_amd.solver import MGPCG
    k = np.exp(np.random.default_rng(7).uniform(-1.0, 1.0, 1 << (2 * lvl))) if coef else None
    H = pb.hierarchy(dim, deg, lvl, 1, kcell=k)
    d = np.random.default_rng(5).integers(-1000, 1000, H.n).astype(np.float64)
    d[H.levels[0].bnd] = 0.0
    out = []
    for inner in ("f64", "f32"):
        s = MGPCG(H, inner=inner, cycle=cycle).init()
        assert s.info()["tail_levels"] == lvl
        c = torch.empty(H.n, dtype=torch.float64, device="cuda")
        s.vcycle(c, torch.from_numpy(d).cuda())
        out.append(c.cpu().numpy())
        s.done()
    err = np.linalg.norm(out[1] - out[0]) / np.linalg.norm(out[0])
    print(f"  {dim}D Q{deg} level {lvl} {cycle} coefficient {coef}: {err * 2 ** 24:.3f} u", flush=True)
    assert err <= 1.001 * 2.0 ** -24


@pytest.mark.parametrize("inner,cells,matrices", [("f64", 44, 0), ("f32", 44, 1), ("f64", 40, 1), ("f32", 64, 0)])
def test_tails_that_keep_their_steps(torch, inner, cells, matrices):
    """A tail of 2025 rows whose vectors with twice the digits exceed the LDS in FP64, and one of 4225 rows,
    run step by step; with 1681 rows FP64 has its matrix too.  Against the launches level by level."""
    from feat3_amd.solver import MGPCG
    from test_gpu_lattice import lattice_hierarchy
    H = lattice_hierarchy(2, 1, cells)
    d = np.random.default_rng(5).uniform(-1.0, 1.0, H.n)
    d[H.levels[0].bnd] = 0.0
    dd = torch.from_numpy(d).cuda()
    out = []
    for tail in (4300, 0):
        s = MGPCG(H, inner=inner, options={"tail_max_n": tail}).init()
        info = s.info()
        if tail:
            assert info["tail_levels"] == len(H.levels) and info["tail_matrices"] == matrices, info
        c = torch.empty_like(dd)
        s.vcycle(c, dd)
        out.append(c.cpu().numpy())
        s.done()
    err = np.linalg.norm(out[0] - out[1]) / np.linalg.norm(out[1])
    assert err <= (1e-12 if inner == "f64" else 64 * np.finfo(np.float32).eps)
