"""The tile schedule of the SpMM (dense operand through LDS, output rows in registers) against the CPU oracle: every row in
CSR order with one fma per edge from the old out value, so equal bit for bit.  Forced at small sizes, where the last tile,
the last row block and the last feature slice are ragged."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from _util import random_csr

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _plan(M, K, deg, seed, **kw):
    from super_gnn_amd import supergnn_ops as ops
    rowptr, col, val = random_csr(M, K, deg, seed=seed, **kw)
    return rowptr, col, val, ops.SpmmPlan(torch.from_numpy(rowptr).to(DEV), torch.from_numpy(col).to(DEV), K)


@pytest.mark.parametrize("M,K,F,deg,kw", [
    (1, 1, 1, 3, {}),                                   # one row, one column
    (5, 103, 64, 7, {}), (5, 104, 65, 7, {}), (5, 105, 63, 7, {}),   # either side of one tile and one slice
    (300, 624, 128, 40, {}), (300, 625, 100, 40, {}),   # as many tiles as the ring has, and one more
    (1545, 2000, 192, 60, {}), (1546, 2000, 602, 25, {}),   # either side of a row block of 15 * 103
    (700, 9000, 130, 9, {"empty_frac": 0.3}),           # waves that skip tiles, rows without edges
    (400, 60000, 32, 3, {}),                            # most tiles without an edge: hundreds entered at once
    (2000, 1500, 96, 80, {"hubs": 5, "hub_deg": 1400}),     # very long rows beside short ones
    (900, 700, 70, 30, {"dup": False, "empty_frac": 0.9}),
    (40, 300, 602, 0, {}),                              # no edge at all
])
def test_tile_schedule_bit_identical_to_oracle(M, K, F, deg, kw, monkeypatch):
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    rowptr, col, val, plan = _plan(M, K, deg, M + K + F, **kw)
    rng = np.random.default_rng(F)
    x, init = rng.standard_normal((K, F), dtype=np.float32), rng.standard_normal((M, F), dtype=np.float32)
    w, xd = torch.from_numpy(val).to(DEV), torch.from_numpy(x).to(DEV)
    deg_f = np.maximum(np.diff(rowptr), 1).astype(np.float32)
    assert (plan.tiles(F)[0] > 0) == (col.size > 0)

    want = init.copy(); orc.spmm_accumulate(rowptr, col, val, x, want)
    for _ in range(2):                                  # values taken from the array, then bound
        out = torch.from_numpy(init.copy()).to(DEV)
        plan.run(w, xd, out, accumulate=True)
        assert np.array_equal(out.cpu().numpy(), want)
    assert plan.tiles(F)[1] == (1 if col.size else 0)

    want = np.zeros_like(init); orc.spmm_accumulate(rowptr, col, np.ones_like(val), x, want)
    orc.row_divide(want, deg_f)
    out = torch.from_numpy(init.copy()).to(DEV)
    plan.run(None, xd, out, accumulate=False, row_div=torch.from_numpy(deg_f).to(DEV))
    assert np.array_equal(out.cpu().numpy(), want), "unit weights, overwrite, mean"

    val2 = val + 1                                      # other values after ones
    want = init.copy(); orc.spmm_accumulate(rowptr, col, val2, x, want)
    out = torch.from_numpy(init.copy()).to(DEV)
    plan.run(torch.from_numpy(val2).to(DEV), xd, out, accumulate=True)
    assert np.array_equal(out.cpu().numpy(), want), "rebound"


def test_padding_edges_touch_no_row(monkeypatch):
    """A wave's last batch is filled up with edges into a register that is no row's: operand rows of infinities and NaN that
    no edge names must not reach any row."""
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    M, K, F = 200, 500, 80
    rowptr, col, val, plan = _plan(M, K, 6, 3)
    x = np.random.default_rng(0).standard_normal((K, F), dtype=np.float32)
    unused = np.setdiff1d(np.arange(K), col)
    assert unused.size
    x[unused[::2]], x[unused[1::2]] = np.inf, np.nan
    want = np.zeros((M, F), np.float32); orc.spmm_accumulate(rowptr, col, val, x, want)
    out = torch.full((M, F), 7.0, device=DEV)
    plan.run(torch.from_numpy(val).to(DEV), torch.from_numpy(x).to(DEV), out, accumulate=False)
    assert np.isfinite(want).all() and np.array_equal(out.cpu().numpy(), want)


def test_default_rule_takes_tiles_for_dense_matrices_alone():
    from super_gnn_amd import supergnn_ops as ops, synth
    rp, cl = synth.sbm_graph(40000, 8, 0.05, 0.0025, seed=3, device=DEV)           # about 340 edges per row
    dense = ops.SpmmPlan(rp, cl, 40000)          # rows of more than 128 edges, three bands
    assert dense.tiles(602)[0] > 0 and dense.schedule(602)["band"] == 1
    x = torch.randn(40000, 602, generator=torch.Generator().manual_seed(1)).to(DEV)
    out = torch.zeros(40000, 602, device=DEV)
    dense.run(None, x, out, accumulate=True)
    rows = slice(20000, 20300)
    rpn = rp.cpu().numpy().astype(np.int64)
    lo, hi = rpn[rows.start], rpn[rows.stop]
    want = np.zeros((300, 602), np.float32)
    orc.spmm_accumulate(rpn[rows.start:rows.stop + 1] - lo, cl[lo:hi].cpu().numpy().astype(np.int64), np.ones(hi - lo, np.float32),
                        x.cpu().numpy(), want)
    assert dense.tiles(602)[1] == 1 and np.array_equal(out[rows].cpu().numpy(), want)
    rp, cl = synth.rmat_graph(200000, 2500000, seed=1, device=DEV)
    assert ops.SpmmPlan(rp, cl, 200000).tiles(602)[0] == 0


@pytest.mark.parametrize("F", [1, 511, 512, 513, 2049, 30000, 40001])
def test_rule_answers_for_every_width(F):
    """Long rows in a dense matrix: the rule asks what the band schedule would do, whose windows are 512 columns wide."""
    plan = _plan(600, 500, 60, 11, hubs=3, hub_deg=450)[3]
    assert plan.tiles(F)[0] == 0


def test_unsorted_rows_keep_the_other_schedules(monkeypatch):
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    rowptr, col, val, plan = _plan(300, 400, 50, 9, dup=True)
    x = np.random.default_rng(1).standard_normal((400, 64), dtype=np.float32)
    want = np.zeros((300, 64), np.float32); orc.spmm_accumulate(rowptr, col, val, x, want)
    out = torch.zeros(300, 64, device=DEV)
    plan.run(torch.from_numpy(val).to(DEV), torch.from_numpy(x).to(DEV), out)
    assert plan.tiles(64) == (0, 0) and np.array_equal(out.cpu().numpy(), want)    # rows of at most 128 edges: CSR order


def test_strided_rows_replay_and_calls_that_may_not_allocate(monkeypatch):
    """A captured product replays with the program's own work between; rows may lie at a pitch; a call that may not allocate takes
    the streams once they are there."""
    from super_gnn_amd._lib import check, lib
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    M, K, F = 900, 1300, 130
    rowptr, col, val, plan = _plan(M, K, 50, 5)
    w = torch.from_numpy(val).to(DEV)
    wide_x, wide_out = torch.randn(K, F + 5, device=DEV), torch.zeros(M, F + 3, device=DEV)
    x, out = wide_x[:, 2:2 + F], wide_out[:, 1:1 + F]
    st = torch.cuda.current_stream

    def run(entry, F, x, out):
        check(entry(plan._h, w.data_ptr(), x.data_ptr(), out.data_ptr(), F, x.stride(0), out.stride(0), 0, None, st().cuda_stream))

    run(lib.sgnn_spmm_csr_f32_noalloc, F, x, out)          # nothing built yet: the other schedules
    assert plan.tiles(F)[1] == 0
    run(lib.sgnn_spmm_csr_f32, F, x, out)
    want = np.zeros((M, F), np.float32); orc.spmm_accumulate(rowptr, col, val, x.cpu().numpy(), want)
    assert np.array_equal(out.cpu().numpy(), want)
    wide_out.zero_()
    run(lib.sgnn_spmm_csr_f32_noalloc, F, x, out)
    assert np.array_equal(out.cpu().numpy(), want) and not wide_out[:, 0].any() and not wide_out[:, 1 + F:].any()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(lib.sgnn_spmm_csr_f32, F, x, out)
    for i in range(3):
        wide_x.mul_(1.5)
        wide_out.zero_()
        graph.replay()
        want = np.zeros((M, F), np.float32); orc.spmm_accumulate(rowptr, col, val, x.cpu().numpy(), want)
        assert np.array_equal(out.cpu().numpy(), want), i
        torch.cuda.synchronize()
