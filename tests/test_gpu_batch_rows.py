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
        x = torch.from_numpy(x0).cuda()
        s.correct(x, torch.from_numpy(np.ascontiguousarray(B)).cuda())
        out.append((x.cpu().numpy(), np.array([s.history(k) for k in range(nsys)])))
        s.done()
    assert np.isfinite(out[1][0]).all()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0])
