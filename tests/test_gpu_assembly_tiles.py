"""Device assembly of Q1 values in the plane (k_assemble_q1_2d: tiles of 64 nodes and 4 or 16 fields) against
the host setup, bit for bit: node lines of 2 to 129 (one and several tiles, remainders), 1 to 33 fields,
and rows whose graph is not the nine neighbours in ascending order, which take the general route."""
import ctypes

import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,nfields", [(1, 1), (2, 16), (5, 17), (6, 3), (6, 33), (7, 16), (7, 7), (8, 20)])
def test_tiles_are_bitwise_host_assembly(torch_cuda, level, nfields):
    from feat3_amd.autograd import DiffusionProblem
    torch = torch_cuda
    print(f"case assembly tiles L{level} fields {nfields}", flush=True)
    prob = DiffusionProblem(dim=2, degree=1, level=level)
    K = np.random.default_rng(level * 50 + nfields).uniform(0.1, 10.0, (nfields, 4 ** level))
    dev = prob.assemble(torch.from_numpy(K).cuda())
    Hs = pb.field_hierarchies(2, level, K, 1, 1)
    for i in range(len(Hs[0].levels)):
        host = pb.stacked_values([H.levels[i].A for H in Hs]).reshape(-1)
        assert np.array_equal(dev[i].cpu().numpy(), host), i


def test_other_graphs_take_the_general_route(torch_cuda):
    from feat3_amd import capi
    from feat3_amd.autograd import DiffusionProblem
    torch = torch_cuda
    print("case assembly with another graph", flush=True)
    prob = DiffusionProblem(dim=2, degree=1, level=4)
    A = prob.H.levels[0].A
    K = np.random.default_rng(3).uniform(0.1, 10.0, (5, 256))
    kf = torch.from_numpy(K).cuda()
    ref = prob.assemble(kf)[0].cpu().numpy().reshape(A.nnz, 5)
    col = np.array(A.col_ind)
    e0 = int(A.row_ptr[8 * 17 + 8])
    col[[e0, e0 + 8]] = col[[e0 + 8, e0]]      # the row's first and last columns change places
    rp, ci = torch.from_numpy(A.row_ptr.view(np.int32)).cuda(), torch.from_numpy(col.view(np.int32)).cuda()
    val = torch.empty(A.nnz * 5, dtype=torch.float64, device="cuda")
    capi.call("feat3_assemble_laplace_fields", ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), 2, 1, 4, 5,
              ctypes.c_void_p(prob.ref.ctypes.data), ctypes.c_void_p(kf.data_ptr()), ctypes.c_void_p(rp.data_ptr()),
              ctypes.c_void_p(ci.data_ptr()), A.rows, ctypes.c_void_p(val.data_ptr()))
    out = val.cpu().numpy().reshape(A.nnz, 5)
    want = ref.copy()
    want[[e0, e0 + 8]] = want[[e0 + 8, e0]]
    assert np.array_equal(out, want)
