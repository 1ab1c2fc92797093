"""sgnn_spmm_plan_stack against the parts' own products, bit for bit: parts whose long rows are regrouped by column class,
parts whose long rows are not, parts without any and parts without edges, in every mixture; fp32 with the values unbound and
bound, and fused over packed rows whose segments need row slots."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

#              rows, columns, degrees (dealt out in turn)
SHAPES = {"hubs": (301, 900, [3, 0, 700, 17, 130, 1]), "dense": (64, 333, [129, 333, 200]), "short": (500, 450, [0, 5, 128, 1, 33]),
          "empty": (40, 60, [0]), "one": (1, 2000, [2000])}


def _part(kind, regrouped, seed, monkeypatch):
    from super_gnn_amd import supergnn_ops as ops
    M, K, degrees = SHAPES[kind]
    rng = np.random.default_rng(seed)
    deg = np.minimum(np.resize(degrees, M), K)
    rowptr = np.concatenate([[0], np.cumsum(deg)])
    col = np.concatenate([np.sort(rng.choice(K, d, replace=False)) for d in deg]) if rowptr[-1] else np.zeros(0)
    value = torch.from_numpy(rng.standard_normal(int(rowptr[-1]), dtype=np.float32)).cuda()
    monkeypatch.setenv("SGNN_SPMM_PARTITION", str(int(regrouped)))
    plan = ops.SpmmPlan(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col.astype(np.int64)).cuda(), K)
    monkeypatch.delenv("SGNN_SPMM_PARTITION")
    assert plan.info()["partitioned"] == int(regrouped and bool((deg > 128).any())), kind
    assert plan.info()["long_edges"] == int(deg[deg > 128].sum())
    return plan, value


MIXTURES = [[("hubs", True), ("dense", False), ("short", True), ("hubs", False), ("empty", False), ("one", True)],
            [("dense", False), ("short", False), ("hubs", True)],
            [("hubs", False), ("empty", False), ("dense", False), ("one", False)],
            [("one", True), ("dense", True), ("hubs", True)],
            [("short", False), ("short", True), ("empty", True)]]


@pytest.mark.parametrize("mixture", range(len(MIXTURES)))
def test_stack_equals_its_parts(mixture, monkeypatch):
    from super_gnn_amd import supergnn_ops as ops
    parts = [_part(kind, regrouped, i, monkeypatch) for i, (kind, regrouped) in enumerate(MIXTURES[mixture])]
    plans, values = [p for p, _ in parts], [v for _, v in parts]
    stacked, value = ops.SpmmPlan.stack(plans), torch.cat(values)
    info = stacked.info()
    for key in ("M", "K", "nnz", "long_rows", "pieces", "long_edges"):
        assert info[key] == sum(p.info()[key] for p in plans), key
    assert info["partitioned"] == max(p.info()["partitioned"] for p in plans)
    g = torch.Generator(device="cuda").manual_seed(mixture)
    for F in (100, 33, 260):
        x = torch.randn(stacked.K, F, generator=g, device="cuda")
        init = torch.randn(stacked.M, F, generator=g, device="cuda")
        for accumulate in (True, False, True):   # unbound, bound, bound
            want, got = init.clone(), init.clone()
            row = column = 0
            for p, v in parts:
                p.run(v, x[column:column + p.K], want[row:row + p.M], accumulate=accumulate)
                row, column = row + p.M, column + p.K
            stacked.run(value, x, got, accumulate=accumulate)
            assert torch.equal(got, want), (F, accumulate)
        assert stacked._bound is not None
    F = 64
    for bits in (8, 4, 2):
        cuts = [c for p in plans for c in (p.K // 3, p.K)]   # two segments a part, mostly not whole groups of rows
        base = np.repeat(np.concatenate([[0], np.cumsum([p.K for p in plans])[:-1]]), 2)
        ranges = torch.tensor([0, *(np.asarray(cuts) + base)], dtype=torch.int32)
        x = torch.randn(stacked.K, F, generator=g, device="cuda")
        params = torch.empty(stacked.K, 2, device="cuda")
        segs = ops.quant_segments(ranges, bits)
        data = torch.empty(segs.n_packed, F, dtype=torch.uint8, device="cuda")
        ops.quantize_tensor_for_all_procs(x, data, params, ranges, ranges.numel() - 1, bits)
        init = torch.randn(stacked.M, F, generator=g, device="cuda")
        for _ in range(2):
            want, got = init.clone(), init.clone()
            row = column = packed = 0
            for p, v in parts:
                mine = torch.tensor([0, p.K // 3, p.K], dtype=torch.int32)
                s = ops.quant_segments(mine, bits)
                p.run_quantized(v, data[packed:packed + s.n_packed], params[column:column + p.K], s, bits, want[row:row + p.M])
                row, column, packed = row + p.M, column + p.K, packed + s.n_packed
            stacked.run_quantized(value, data, params, segs, bits, got)
            assert torch.equal(got, want), bits


def test_refused():
    from super_gnn_amd import supergnn_ops as ops
    rowptr, col = torch.tensor([0, 1]).cuda(), torch.tensor([0]).cuda()
    a, b = ops.SpmmPlan(rowptr, col, 1), ops.SpmmPlan(rowptr, col, 1, long_row_threshold=7)
    with pytest.raises(ValueError, match="thresholds"):
        ops.SpmmPlan.stack([a, b])
    with pytest.raises(ValueError, match="itself stacked"):
        ops.SpmmPlan.stack([a, ops.SpmmPlan.stack([a, a])])
