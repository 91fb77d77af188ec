"""The streaming CSR product (k_csr_stream) on both sides of its dispatch: matrices up to 256 MB read eight
products ahead of their sums, larger ones one at a time.  Every row's terms are added in the same order,
so the rows of a large matrix equal, bit for bit, those of a small one that holds them alone; the small
one is checked against FP64 sums (rows of 0 to 47 entries, all remainders of eight among them; error
of a sum of w terms at most (w + 2) eps of the terms' sizes)."""
import numpy as np
import pytest

from feat3_amd import problems as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_large_and_small_matrices_sum_alike(torch_cuda, dtype):
    from feat3_amd import lafem
    torch = torch_cuda
    print(f"case streaming CSR {dtype}", flush=True)
    dt = getattr(torch, dtype)
    size = 12 if dtype == "float64" else 8
    rows, part = (1_000_003, 40_001) if dtype == "float64" else (1_450_007, 40_001)
    rng = np.random.default_rng(1)
    n = rng.integers(0, 48, rows)
    rp = np.concatenate([[0], np.cumsum(n)])
    assert rp[-1] * size > 1 << 28 > rp[part] * size
    col = ((np.repeat(np.arange(rows), n) + 7919 * (np.arange(rp[-1]) - np.repeat(rp[:-1], n))) % rows).astype(np.uint32)
    val = rng.uniform(-1.0, 1.0, rp[-1])
    x = rng.uniform(-1.0, 1.0, rows)
    y = rng.uniform(-1.0, 1.0, rows)
    out = []
    for k in (rows, part):
        A = lafem.SparseMatrixCSR(pb.Csr(k, rows, rp[: k + 1].astype(np.uint32), col[: rp[k]], val[: rp[k]]), dtype=dt)
        r = lafem.DenseVector(k, dt)
        A.apply(r, lafem.DenseVector(torch.from_numpy(x).cuda().to(dt)), lafem.DenseVector(torch.from_numpy(y[:k].copy()).cuda().to(dt)), -0.5)
        out.append(r.t.cpu().numpy())
    assert np.array_equal(out[0][:part], out[1])
    f = np.dtype(dtype).type
    v, xs, ys = (a.astype(f).astype(np.float64) for a in (val[: rp[part]], x, y[:part]))
    row = np.repeat(np.arange(part), n[:part])
    terms = v * xs[col[: rp[part]].astype(np.int64)]
    exact = ys - 0.5 * np.bincount(row, terms, part)
    size_of = np.abs(ys) + 0.5 * np.bincount(row, np.abs(terms), part)
    assert (np.abs(out[1] - exact) <= 50 * np.finfo(f).eps * size_of).all()
