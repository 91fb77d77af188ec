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
        c = torch.empty_like(dd)
        for _ in range(2):      # a second cycle starts from the first one's buffers
            s.vcycle(c, dd)
        out.append(c.cpu().numpy())
        s.done()
    err = np.linalg.norm(out[0] - out[1]) / np.linalg.norm(out[1])
    print(f"  {dim}D Q{deg} level {lvl} {cycle} {inner}: {err:.2e}", flush=True)
    assert err <= (1e-12 if inner == "f64" else 64 * np.finfo(np.float32).eps)
