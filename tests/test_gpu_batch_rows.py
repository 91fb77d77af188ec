"""Several steps of a level with one matrix per system in one pass (batch_rows.hpp) against one launch per
step (option lattice = 0): every sum takes the same terms in the same order, and no reduction is
involved, so whole solves agree bit for bit."""
import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("level,nsys,pre,post", [(7, 1, 4, 4), (7, 3, 1, 1), (7, 16, 4, 4), (7, 17, 2, 3), (7, 20, 3, 5),
                                                 (7, 40, 5, 2), (8, 5, 4, 4), (8, 16, 2, 6), (9, 2, 4, 4)])
def test_rows_match_single_steps(torch_cuda, inner, level, nsys, pre, post):
    from feat3_amd.batch import BatchMGPCG
    torch = torch_cuda
    print(f"case rows {inner} L{level} K={nsys} {pre}+{post}", flush=True)
    H = pb.hierarchy(2, 1, level, 1)
    rng = np.random.default_rng(level * 100 + nsys)
    # symmetric positive definite: every system scales the Laplacian of each node pair differently
    vals = []
    for L in H.levels:
        n = L.A.row_ptr.size - 1
        rows = np.repeat(np.arange(n), np.diff(L.A.row_ptr.astype(np.int64)))
        w = rng.uniform(0.8, 1.25, (n, nsys))
        vals.append(np.ascontiguousarray(np.asarray(L.A.val)[:, None] * w[rows] * w[L.A.col_ind.astype(np.int64)]))
    B = pb.random_rhs(H.n, 1, nsys, H.levels[0].bnd, seed=5)
    x0 = np.random.default_rng(6).standard_normal(B.shape)   # boundary values included
    out = []
    for lattice in (1, 0):
        s = BatchMGPCG(H, nsys, values=vals, shared=False, inner=inner, pre=pre, post=post, tol_rel=0.0, min_iter=3,
                       max_iter=3, options={"lattice": lattice}).init()
        info = s.info()      # the route: levels of 100 nodes per axis or more
        assert info["pass_levels"] == (level - 6 if lattice else 0)
        assert info["steps_per_pass"] == ({"f64": 2, "f32": 4, "f16": 3}[inner] if lattice else 0)
        x = torch.from_numpy(x0).cuda()
        s.correct(x, torch.from_numpy(np.ascontiguousarray(B)).cuda())
        out.append((x.cpu().numpy(), np.array([s.history(k) for k in range(nsys)])))
        s.done()
    assert np.isfinite(out[1][0]).all()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,level,nsys,tail", [(2, 4, 1, 300), (2, 5, 16, 1100), (2, 6, 5, 1100), (2, 6, 16, 4300), (3, 3, 3, 800),
                                                 (2, 3, 40, 5000)])
def test_field_tail_is_identical(torch_cuda, inner, dim, level, nsys, tail):
    """One matrix per system: the levels of at most tail_max_n nodes in one workgroup per system against
    the per-level launches (tail_max_n 0), bit for bit; also after new values (every level's copies)."""
    import ctypes
    from feat3_amd import capi
    from feat3_amd.batch import BatchMGPCG
    torch = torch_cuda
    print(f"case field tail {inner} {dim}D L{level} K={nsys} tail {tail}", flush=True)
    H = pb.hierarchy(dim, 1, level, 1)
    rng = np.random.default_rng(level * 10 + nsys)
    sets = [[np.ascontiguousarray(np.asarray(L.A.val)[:, None] * rng.uniform(0.5, 2.0, nsys)) for L in H.levels] for _ in range(2)]
    B = torch.from_numpy(np.ascontiguousarray(pb.random_rhs(H.n, 1, nsys, H.levels[0].bnd, seed=5))).cuda()
    out = []
    for t in (tail, 0):
        s = BatchMGPCG(H, nsys, values=sets[0], shared=False, inner=inner, options={"tail_max_n": t}).init()
        # the deepest levels within the limit whose five vectors fit 160 KB of LDS
        used, want = 0, 0
        for L in reversed(H.levels):
            used += 5 * L.A.rows * (8 if inner == "f64" else 4)
            if want and (L.A.rows > t or used > 160 * 1024):
                break
            want += 1
        assert s.info()["tail_levels"] == (want if want > 1 else 0)
        res = []
        for new in (False, True):
            if new:
                dev = [torch.from_numpy(v).cuda() for v in sets[1]]
                for i, v in enumerate(dev):
                    capi.call("feat3_batch_set_values", s._h, i, ctypes.c_void_p(v.data_ptr()))
            x = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
            st, it = s.correct(x, B)
            assert (st == 2).all()
            res += [x.cpu().numpy(), it, np.concatenate([s.history(k) for k in range(nsys)])]
        out.append(res)
        s.done()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("case", ["q1", "weight"])
def test_lattice_prolongation_is_identical(torch_cuda, case):
    """The prolongation by its closed form against the stored matrix, bit for bit; a matrix with one other
    weight keeps the stored one (7 systems: one value per thread, 8: four)."""
    from feat3_amd.batch import BatchMGPCG
    torch = torch_cuda
    for nsys in (7, 8):
        print(f"case lattice prolongation {case} K={nsys}", flush=True)
        H = pb.hierarchy(2, 1, 7, 1)
        if case == "weight":
            H.levels[0].P.val = np.array(H.levels[0].P.val)
            H.levels[0].P.val[int(H.levels[0].P.row_ptr[64 * 129 + 65])] = 0.375
        vals = [np.ascontiguousarray(np.repeat(np.asarray(L.A.val)[:, None], nsys, axis=1)) for L in H.levels]
        B = torch.from_numpy(np.ascontiguousarray(pb.random_rhs(H.n, 1, nsys, H.levels[0].bnd, seed=5))).cuda()
        out = []
        for lattice in (1, 0):
            s = BatchMGPCG(H, nsys, values=vals, shared=False, inner="f32", tol_rel=0.0, min_iter=2, max_iter=2,
                           options={"lattice": lattice}).init()
            assert s.info()["lattice_prolongations"] == (1 if lattice and case == "q1" else 0)
            x = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
            s.correct(x, B)
            out.append(x.cpu().numpy())
            s.done()
        assert np.isfinite(out[1]).all() and np.array_equal(out[0], out[1])
