"""The batched solver's values: new ones of every level (feat3_batch_set_values) between two solves into the
SAME solution vector, and ones that are not finite.

The second solve replays the iterations captured by the first one, whose launches hold device addresses;
what they read (the coarse inverses among it) is refreshed in place.  The solution has to be, bit for
bit, that of a solver built for the new values.  Allocations made in between take whatever memory the
refresh would have given back."""
import ctypes

import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inner", ["f64", "f32"])
@pytest.mark.parametrize("nsys,shared,tail", [(3, False, 1100), (16, False, 0), (4, True, 1000), (4, True, 0)])
def test_replayed_iterations_take_the_new_values(torch_cuda, inner, nsys, shared, tail):
    from feat3_amd import capi
    from feat3_amd.batch import BatchMGPCG
    torch = torch_cuda
    print(f"case new values {inner} K={nsys} shared={shared} tail {tail}", flush=True)
    H = pb.hierarchy(2, 1, 5, 1)
    rng = np.random.default_rng(nsys)
    f = [rng.uniform(0.5, 2.0, 1 if shared else nsys) for _ in range(3)]
    sets = [[np.ascontiguousarray(np.asarray(L.A.val)[:, None] * w) for L in H.levels] for w in f]
    B = torch.from_numpy(np.ascontiguousarray(pb.random_rhs(H.n, 1, nsys, H.levels[0].bnd, seed=5))).cuda()

    def make(vals):
        return BatchMGPCG(H, nsys, values=vals, shared=shared, inner=inner, options={"tail_max_n": tail}).init()

    s = make(sets[0])
    x = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
    s.correct(x, B)
    held = []
    for vals in sets[1:] + sets[:1]:
        for i, v in enumerate(vals):
            dv = torch.from_numpy(v).cuda()
            capi.call("feat3_batch_set_values", s._h, i, ctypes.c_void_p(dv.data_ptr()))
            held += [dv, torch.full((1 << 16,), float("nan"), dtype=torch.float64, device="cuda")]
        x.zero_()
        st, it = s.correct(x, B)
        e = make(vals)
        y = torch.zeros_like(x)
        se, ie = e.correct(y, B)
        e.done()
        assert (st == 2).all() and (se == 2).all() and (it == ie).all()
        assert torch.equal(x, y)
    s.done()


@pytest.mark.parametrize("inner", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,lvl,shared,block", [(2, 7, False, 1), (3, 3, True, 1), (3, 3, True, 3)])
def test_dirichlet_rows_that_are_not_finite(torch_cuda, dim, lvl, shared, block, inner):
    """A NaN or an infinity in the matrix row of a Dirichlet node, at init or in new values: every system
    that has it ends with status aborted and the others are solved, as with the row kernels (lattice = 0)."""
    from feat3_amd import capi
    from feat3_amd.batch import BatchMGPCG
    torch = torch_cuda
    print(f"case Dirichlet rows {inner} {dim}D L{lvl} shared={shared} B={block}", flush=True)
    H = pb.hierarchy(dim, 1, lvl, 1)
    nsys = 4
    B = torch.from_numpy(np.ascontiguousarray(pb.random_rhs(H.n, block, nsys, H.levels[0].bnd, seed=5))).cuda()

    def values(level=None, bad=None):
        if block == 3:
            v = [pb.block_identity_values(L.A, 3) for L in H.levels]
        else:
            v = [np.repeat(np.asarray(L.A.val)[:, None], 1 if shared else nsys, axis=1) for L in H.levels]
        if level is not None:
            L = H.levels[level]
            e = int(L.A.row_ptr[int(L.bnd[L.bnd.size // 3])])
            (v[level] if block == 3 else v[level][:, -1])[e] = bad
        return [np.ascontiguousarray(a) for a in v]

    for level, bad in ((0, np.nan), (0, np.inf), (1, np.nan)):
        out = []
        for lattice in (1, 0):
            s = BatchMGPCG(H, nsys, values=values(level, bad), block=block, shared=shared, inner=inner,
                           options={"lattice": lattice, "tail_max_n": 0 if shared else 1100}).init()
            x = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
            out.append([a.tolist() for a in s.correct(x, B)])
            s.done()
        assert out[0] == out[1], (level, bad, out)
        assert out[0][0] == ([3] * nsys if shared else [2, 2, 2, 3])
        if not shared:
            s = BatchMGPCG(H, nsys, values=values(), shared=False, inner=inner).init()
            x = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
            assert (s.correct(x, B)[0] == 2).all()
            for vals, want in ((values(level, bad), [2, 2, 2, 3]), (values(), [2] * nsys)):
                for i, v in enumerate(vals):
                    dv = torch.from_numpy(v).cuda()
                    capi.call("feat3_batch_set_values", s._h, i, ctypes.c_void_p(dv.data_ptr()))
                x.zero_()
                assert s.correct(x, B)[0].tolist() == want
            s.done()
