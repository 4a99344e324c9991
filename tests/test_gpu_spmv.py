"""The standalone block SpMV on the GPU at the edges of its row groups: fewer
rows than a workgroup, one more, rows without blocks, rows of more blocks
than one pass takes (16), and each lane count, against FP64.

Tolerance: a row is a sum of at most 3 (len + 1) FP32 products in any order,
so its error is at most (3 (len + 1) + 2) 2^-24 times the sum of their sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [4, 8, 16])
@pytest.mark.parametrize("n", [1, 15, 17, 33, 64, 65, 1000])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.5, 2.0)])
def test_spmv_rows(gpu, n, lanes, alpha, beta):
    import torch

    from chysx import abi

    rng = np.random.default_rng(31 * n + lanes)
    lens = rng.choice([0, 1, 3, 7, 8, 9, 12, 16, 17, 32, 41], n)
    lens[n - 1] = 17
    ro = np.zeros(n + 1, np.int32)
    np.cumsum(lens, out=ro[1:])
    ci = rng.integers(0, n, ro[-1]).astype(np.int32)
    val = rng.normal(size=(ro[-1], 3, 3)).astype(np.float32)
    diag = rng.normal(size=(n, 3, 3)).astype(np.float32)
    x, y0 = rng.normal(size=(2, n, 3)).astype(np.float32)
    rows = np.repeat(np.arange(n), lens)
    want = np.einsum("nij,nj->ni", diag.astype(np.float64), x.astype(np.float64))
    size = np.einsum("nij,nj->ni", np.abs(diag).astype(np.float64), np.abs(x).astype(np.float64))
    np.add.at(want, rows, np.einsum("nij,nj->ni", val.astype(np.float64), x[ci].astype(np.float64)))
    np.add.at(size, rows, np.einsum("nij,nj->ni", np.abs(val).astype(np.float64), np.abs(x[ci]).astype(np.float64)))
    want = alpha * want + beta * y0
    bound = (3 * (lens[:, None] + 1) + 4) * 2.0**-24 * (abs(alpha) * size + abs(beta) * np.abs(y0)) + 1e-30
    t = [torch.from_numpy(a).cuda() for a in (diag, ro, ci, val, x, y0)]
    abi.spmv_bsr3(n, *(a.data_ptr() for a in t), alpha, beta, lanes)
    torch.cuda.synchronize()
    assert (np.abs(t[5].cpu().numpy() - want) <= bound).all()
