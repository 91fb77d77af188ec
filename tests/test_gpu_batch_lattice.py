"""The batched solver's steps by lines (batch_lattice.hpp) against its row kernels (option lattice = 0).

Every row sum takes the same terms in the same order, so the cycles agree bit for bit; the outer
product's partial sums are grouped by other blocks.  A dot product of n FP64 terms regrouped differs by
at most n eps relative to the sum of the terms' sizes; p.q and the squared norms are sums of (nearly)
positive terms, so the scalars of an iteration differ by less than n eps (n <= 5e4 here: 1e-11), which
an iteration carries on with a factor near one.  A term taken wrongly, or summed in another order in FP32
(1e-7), shows far above that.
"""
import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


def solve(torch, H, B, nsys, vals, block, inner, lattice, x0=None, iters=4):
    from feat3_amd.batch import BatchMGPCG
    s = BatchMGPCG(H, nsys, values=vals, block=block, inner=inner, tol_rel=0.0, min_iter=iters, max_iter=iters,
                   options={"lattice": lattice, "tail_max_n": 0}).init()
    x = torch.zeros(s.shape, dtype=torch.float64, device="cuda") if x0 is None else torch.from_numpy(x0).cuda()
    st, it = s.correct(x, torch.from_numpy(np.ascontiguousarray(B)).cuda())
    h = [s.history(k)[: iters + 1] for k in range(nsys)]
    nbytes = s.time_kernel(0, 1)[1]
    route = {k: s.info()[k] for k in ("line_levels", "outer_lines", "lattice_prolongations")}
    assert lattice or not any(route.values())
    s.done()
    return list(st), list(it), x.cpu().numpy(), np.array(h), nbytes, route


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("level,block,nsys", [(2, 1, 1), (3, 3, 1), (3, 1, 7), (4, 3, 5), (4, 1, 40), (4, 3, 32), (5, 1, 4),
                                              (3, 1, 64)])
def test_lines_match_the_row_kernels(torch_cuda, inner, level, block, nsys):
    torch = torch_cuda
    print(f"case lines {inner} L{level} B={block} K={nsys}", flush=True)
    H = pb.hierarchy(3, 1, level, 1)
    vals = [pb.block_identity_values(L.A, 3) for L in H.levels] if block == 3 else None
    B = pb.random_rhs(H.n, block, nsys, H.levels[0].bnd, seed=5)
    x0 = np.random.default_rng(6).standard_normal(B.shape)   # the initial defect's product, boundary values included
    a = solve(torch, H, B, nsys, vals, block, inner, 1, x0)
    b = solve(torch, H, B, nsys, vals, block, inner, 0, x0)
    assert a[0] == b[0] and a[1] == b[1]
    assert a[4] < b[4]   # the route was taken: no matrix among the sweep's bytes
    assert a[5] == {"line_levels": level - 1, "outer_lines": 1, "lattice_prolongations": level - 1}
    assert np.allclose(a[3], b[3], rtol=1e-10, atol=0)
    assert np.linalg.norm(a[2] - b[2]) <= 1e-10 * np.linalg.norm(b[2])
    assert np.array_equal(a[3][:, 0] > 0, b[3][:, 0] > 0)


@pytest.mark.parametrize("change", ["value", "boundary", "tap"])
def test_unequal_rows_keep_the_row_kernels(torch_cuda, change):
    """One inner row that differs (a value, an explicit Dirichlet row, or an entry of another column)
    sends its level to the row kernels: the results are those of lattice = 0 bit for bit."""
    torch = torch_cuda
    print(f"case lines refused {change}", flush=True)
    H = pb.hierarchy(3, 1, 3, 1)
    L = H.levels[0]
    mid = 4 * 81 + 4 * 9 + 4
    vals = [np.array(l.A.val, np.float64) for l in H.levels]
    e0 = int(L.A.row_ptr[mid])
    if change == "value":
        vals[0][e0 + 13] *= 1.25
    elif change == "boundary":
        L.bnd = np.sort(np.append(L.bnd, np.array([mid], L.bnd.dtype)))
    else:
        L.A.col_ind = np.array(L.A.col_ind)
        L.A.col_ind[e0] = mid - 81 - 9 - 2
    B = pb.random_rhs(H.n, 1, 4, L.bnd, seed=7)
    for inner in ("f64", "f32"):
        a = solve(torch, H, B, 4, vals, 1, inner, 1, iters=2)
        b = solve(torch, H, B, 4, vals, 1, inner, 0, iters=2)
        assert a[4] == b[4] and a[5]["outer_lines"] == 0 and a[5]["line_levels"] == len(H.levels) - 2
        assert np.array_equal(a[3], b[3])
        assert np.linalg.norm(a[2] - b[2]) <= 1e-11 * np.linalg.norm(b[2])


def test_new_values_leave_the_lines(torch_cuda):
    """A level that gets new values (full blocks) runs the row kernels from then on."""
    import ctypes
    from feat3_amd import capi
    from feat3_amd.batch import BatchMGPCG
    torch = torch_cuda
    print("case lines and new values", flush=True)
    H = pb.hierarchy(3, 1, 3, 1)
    vals = [np.array(l.A.val, np.float64) for l in H.levels]
    new = vals[0] * np.random.default_rng(8).uniform(0.9, 1.1, vals[0].size)
    B = torch.from_numpy(pb.random_rhs(H.n, 1, 4, H.levels[0].bnd, seed=9)).cuda()
    out = []
    for lattice in (1, 0):
        s = BatchMGPCG(H, 4, inner="f64", tol_rel=0.0, min_iter=3, max_iter=3, options={"lattice": lattice}).init()
        x = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
        s.correct(x, B)
        lines = s.info()["line_levels"]
        dv = torch.from_numpy(new).cuda()
        capi.call("feat3_batch_set_values", s._h, 0, ctypes.c_void_p(dv.data_ptr()))
        assert s.info()["outer_lines"] == 0 and s.info()["line_levels"] == max(0, lines - 1)
        x.zero_()
        s.correct(x, B)
        out.append(x.cpu().numpy())
        s.done()
    assert np.linalg.norm(out[0] - out[1]) <= 1e-10 * np.linalg.norm(out[1])
