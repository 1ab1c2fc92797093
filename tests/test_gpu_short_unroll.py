"""Short-row kernel: both numbers of gathers in flight, at every lane-group width and at the edges of a group's
32 / 64-edge window, bit for bit against the oracle (rows of up to 128 edges keep the reference's fma order)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _matrix(M, K, degrees, seed):
    rng = np.random.default_rng(seed)
    deg = np.resize(np.asarray(degrees, dtype=np.int64), M)
    rowptr = np.concatenate([[0], np.cumsum(deg)])
    return rowptr, rng.integers(0, K, size=int(rowptr[-1]), dtype=np.int64), rng.standard_normal(int(rowptr[-1]), dtype=np.float32)


# 400 rows give a few hundred chunks (one resident round of waves); 36000 rows of about 33 edges more than 16384 chunks
@pytest.mark.parametrize("M", [400, 36000])
@pytest.mark.parametrize("F", [20, 32, 36, 64, 68, 100, 128, 132, 256])
def test_gathers_in_flight(M, F):
    from super_gnn_amd import supergnn_ops as ops
    K = 500
    rowptr, col, val = _matrix(M, K, [1, 33, 0, 7, 64, 128, 2, 31, 65, 8, 16, 0, 100, 3, 32, 40], seed=F + M)
    rng = np.random.default_rng(F)
    x = rng.standard_normal((K, F), dtype=np.float32)
    div = rng.integers(1, 9, size=M).astype(np.float32)
    plan = ops.SpmmPlan(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), K)
    assert plan.info()["long_rows"] == 0
    v, xg = torch.from_numpy(val).cuda(), torch.from_numpy(x).cuda()
    init = rng.standard_normal((M, F), dtype=np.float32)
    for accumulate, row_div in ((True, None), (False, None), (True, div)):
        want = init.copy() if accumulate else np.zeros_like(init)
        orc.spmm_accumulate(rowptr, col, val, x, want)
        if row_div is not None:
            want = want / row_div[:, None]
        out = torch.from_numpy(init.copy()).cuda()
        plan.run(v, xg, out, accumulate=accumulate, row_div=None if row_div is None else torch.from_numpy(row_div).cuda())
        assert np.array_equal(out.cpu().numpy(), want), (M, F, accumulate, row_div is not None)
