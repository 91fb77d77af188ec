"""One solver, many solution vectors: the captured iteration reads the solution's address from the solver
state, so a solve into another vector (or a view at an odd offset) is the same solve bit for bit, and solves
that end at their first publication leave nothing behind for the next one."""
import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,inner", [("csr", "f64"), ("banded", "f32")])
def test_every_vector_gets_its_solution(fmt, inner):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from feat3_amd.solver import MGPCG
    H = pb.hierarchy(2, 1, 6, 1)
    s = MGPCG(H, inner=inner, fmt=fmt).init()
    b = torch.from_numpy(pb.filtered_rhs(H, 0)).cuda()
    zero = torch.zeros_like(b)
    ref = torch.zeros_like(b)
    st, it = s.correct(ref, b)
    assert st == 2 and it > 1
    buf = torch.zeros(4 * H.n + 7, dtype=torch.float64, device="cuda")
    for k in range(4):
        x = buf[k * (H.n + 1): k * (H.n + 1) + H.n]
        assert s.correct(x, b) == (st, it)
        assert torch.equal(x, ref)
        # converged at the first publication: a zero right-hand side, then a solve again
        y = torch.zeros_like(b)
        assert s.correct(y, zero)[1] == 0 and not y.any()
    assert np.array_equal(ref.cpu().numpy(), buf[: H.n].cpu().numpy())
    s.done()
