"""Short-row kernel: every number of gathers in flight, at every lane-group width, lane width and at the edges of a group's
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


# 400 rows give a few hundred chunks, 36000 rows of about 33 edges 11250
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


def _check(plan, rowptr, col, val, x, xg, rows=None):
    """Overwrite, accumulate and divide against the oracle, on all rows or on a sample of them."""
    M, F = rowptr.size - 1, x.shape[1]
    rng = np.random.default_rng(F)
    v = torch.from_numpy(val).cuda()
    init = rng.standard_normal((M, F), dtype=np.float32)
    div = rng.integers(1, 9, size=M).astype(np.float32)
    rows = np.arange(M) if rows is None else rows
    edges = np.concatenate([np.arange(rowptr[r], rowptr[r + 1]) for r in rows])
    part = np.concatenate([[0], np.cumsum((rowptr[1:] - rowptr[:-1])[rows])])
    for accumulate, row_div in ((False, None), (True, div)):
        want = init[rows].copy() if accumulate else np.zeros((rows.size, F), np.float32)
        orc.spmm_accumulate(part, col[edges], val[edges], x, want)
        if row_div is not None:
            want = want / row_div[rows][:, None]
        out = torch.from_numpy(init.copy()).cuda()
        plan.run(v, xg, out, accumulate=accumulate, row_div=None if row_div is None else torch.from_numpy(row_div).cuda())
        got = out.cpu().numpy()[rows]
        assert np.array_equal(got, want), (M, F, accumulate, row_div is not None)


DEGREES = [1, 33, 0, 7, 64, 128, 2, 31, 65, 8, 16, 0, 100, 3, 32, 40]
# rows, columns, degrees, hubs in front (rows of 3000 edges that make the graph a skewed one), F, rows in flight.
# The row counts stand on both sides of the dispatch's lines: 2048 waves, 10240, 16384 chunks, and the operand's size.
FORMS = [(400, 500, DEGREES, 0, F, 8) for F in (20, 33, 64, 66, 100, 160, 256)] + [
    (60000, 500, DEGREES, 0, 20, 8), (60000, 500, DEGREES, 0, 64, 3), (60000, 500, DEGREES, 0, 100, 2), (60000, 500, DEGREES, 0, 128, 2),
    (60000, 500, DEGREES, 0, 132, 0), (60000, 500, DEGREES, 0, 256, 0), (60000, 500, DEGREES, 0, 50, 2), (60000, 500, DEGREES, 0, 33, 8),
    (60000, 500, DEGREES, 0, 66, 4), (60000, 500, DEGREES, 0, 30, 3), (60000, 500, DEGREES, 0, 13, 8), (60000, 500, DEGREES, 0, 29, 8),
    (15000, 500, [17], 0, 66, 4), (15000, 500, [17], 0, 50, 8), (12000, 500, [17], 12, 66, 8), (60000, 500, DEGREES, 60, 90, 4),
    (9000, 15000, [17], 0, 128, 8), (9000, 16000, [17], 0, 128, 2), (15000, 500, [17], 0, 128, 2),
    (15000, 20000, [17], 0, 160, 8), (15000, 21000, [17], 0, 160, 2), (15000, 500, [17], 0, 164, 2), (5000, 7000, [17], 0, 256, 8),
    (5000, 9000, [17], 0, 256, 2), (15000, 20000, [17], 0, 256, 2), (16000, 22000, [17], 0, 256, 0), (14000, 22000, [17], 0, 256, 2),
    (12000, 500, [17], 12, 128, 8), (12000, 22000, [17], 12, 256, 8), (60000, 500, DEGREES, 60, 100, 2), (60000, 500, DEGREES, 60, 256, 0)]


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"{f[0]}x{f[1]}-hubs{f[3]}-F{f[4]}-{f[5]}")
def test_every_depth_against_the_oracle(form):
    from super_gnn_amd import supergnn_ops as ops
    M, K, degrees, hubs, F, depth = form
    rowptr, col, val = _matrix(M, K, degrees, seed=F + M)
    if hubs:   # long rows in front: they are summed by the piece kernel and not looked at here
        rng = np.random.default_rng(M)
        front = -(-int(col.size) // (7 * 3000)) + hubs   # an eighth of the edges and a few more
        rowptr = np.concatenate([np.arange(front) * 3000, rowptr + front * 3000])
        col = np.concatenate([rng.integers(0, K, size=front * 3000, dtype=np.int64), col])
        val = np.concatenate([rng.standard_normal(front * 3000, dtype=np.float32), val])
    plan = ops.SpmmPlan(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), K)
    chunks, got = plan.short_rows(F)
    assert got == depth, (chunks, got)
    assert (plan.info()["long_edges"] * 8 >= plan.info()["nnz"]) == bool(hubs)
    x = np.random.default_rng(F).standard_normal((K, F), dtype=np.float32)
    rows = np.arange(front, rowptr.size - 1) if hubs else None
    _check(plan, rowptr, col, val, x, torch.from_numpy(x).cuda(), rows)


@pytest.mark.parametrize("F,depth", [(64, 3), (100, 2), (128, 2)])
def test_an_operand_beyond_the_infinity_cache(F, depth):
    """More than 256 MB of dense rows: the launch asks for LDS that it does not use."""
    from super_gnn_amd import supergnn_ops as ops
    K = (260 << 20) // (4 * F)
    rowptr, col, val = _matrix(60000, K, DEGREES, seed=F)
    plan = ops.SpmmPlan(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), K)
    assert plan.short_rows(F)[0] > 16384 and plan.short_rows(F)[1] == depth
    x = np.random.default_rng(F).standard_normal((K, F), dtype=np.float32)
    _check(plan, rowptr, col, val, x, torch.from_numpy(x).cuda(), np.arange(0, 60000, 37))


@pytest.mark.parametrize("F", [100, 160, 256])
def test_rows_on_eight_byte_boundaries(F):
    """The same matrix with an operand and results that start 8 bytes past a 16-byte boundary: two-float lanes."""
    from super_gnn_amd import _lib, supergnn_ops as ops
    for M in (400, 60000):
        rowptr, col, val = _matrix(M, 500, DEGREES, seed=F + M)
        plan = ops.SpmmPlan(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), 500)
        x = torch.randn(500, F, generator=torch.Generator(device="cuda").manual_seed(F), device="cuda")
        v = torch.from_numpy(val).cuda()
        want = torch.empty(M, F, device="cuda")
        plan.run(v, x, want, accumulate=False)
        shifted, out = torch.zeros(500 * F + 2, device="cuda"), torch.zeros(M * F + 2, device="cuda")
        shifted[2:] = x.reshape(-1)
        _lib.check(_lib.lib.sgnn_spmm_csr_f32(plan._h, v.data_ptr(), shifted.data_ptr() + 8, out.data_ptr() + 8, F, F, F, 0, None, ops._stream()))
        assert torch.equal(out[2:].view(M, F), want) and bool((out[:2] == 0).all())
