"""The partitions' stacked matrices against the partitions one by one: the same floats, for every exchange format, both
modes, widths with and without the fused remote step, graphs without and with long rows.  (At these sizes every long row is
regrouped; test_gpu_plan_stack.py mixes regrouped and plain ones.)  Then what the stacked form must not change: edits of the
values, bound or not, seen by a version counter or not; partitions that stacking does not fit; what is refused."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 3501


def _world(P, F, bits, pre, wire):
    from super_gnn_amd import synth
    from super_gnn_amd.aggregator import LoopbackWorld
    from super_gnn_amd.data_manager import build_loopback_partitions
    if P == 5:
        rowptr, col = synth.rmat_graph(N, 16 * N, seed=F)
    else:
        rowptr, col = synth.uniform_degree_graph(N, 7, seed=P + F)
    value = torch.rand(col.numel(), generator=torch.Generator().manual_seed(F))
    graphs = build_loopback_partitions(rowptr, col, value, P, F, num_bits=bits, is_pre_delay=pre)
    return LoopbackWorld(graphs, bits, pre, params_wire_dtype=torch.bfloat16 if wire else None)


def _both(world, x, grad, bits, pre):
    from super_gnn_amd.aggregator import Aggregator, _world_backward, _world_forward
    a = x.clone().requires_grad_()
    out = Aggregator.apply(world, a, 0, bits, pre, True)
    out.backward(grad)
    outs = _world_forward(world, torch.split(x, world.partition_sizes), bits)
    grads = _world_backward(world, torch.split(grad, world.partition_sizes), bits)
    return (out.detach(), a.grad), (torch.cat(outs), torch.cat(grads))


@pytest.mark.parametrize("pre", [False, True])
@pytest.mark.parametrize("bits", [32, 16, 8, 4, 2])
@pytest.mark.parametrize("P,F", [(2, 64), (3, 33), (5, 100), (8, 128)])
def test_stacked_equals_one_by_one(P, F, bits, pre):
    world = _world(P, F, bits, pre, wire=P == 3 and bits < 16)
    g = torch.Generator(device="cuda").manual_seed(1)
    for seed in range(2):
        x = torch.randn(N, F, generator=g, device="cuda")
        grad = torch.randn(N, F, generator=g, device="cuda")
        got, want = _both(world, x, grad, bits, pre)
        # both directions took the stacked products: the first side of the comparison is not the second one again
        assert all(world._stacked.products["local", back].plan is not None and back in world._stacked.spaces for back in (False, True))
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_edited_values_are_seen():
    world = _world(3, 64, 32, True, False)
    g = torch.Generator(device="cuda").manual_seed(2)
    x, grad = (torch.randn(N, 64, generator=g, device="cuda") for _ in range(2))
    before, _ = _both(world, x, grad, 32, True)
    world.graphs[1].local_adj_t.csr()[2].mul_(2)
    got, want = _both(world, x, grad, 32, True)
    assert torch.equal(got[0], want[0]) and not torch.equal(got[0], before[0])
    assert torch.equal(got[1], want[1]) and torch.equal(got[1], before[1])   # the transposed values are a copy of their own


def _mats(world):
    return [m for g in world.graphs for m in (g.local_adj_t, *((g.adj_t_pre_post_aggr_from, g.adj_t_pre_post_aggr_to)
                                                               if world.is_pre_delay else (g.remote_adj_t,)))]


def _same(world, x, grad, bits, pre):
    got, want = _both(world, x, grad, bits, pre)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    return got


@pytest.mark.parametrize("bits", [32, 4])
@pytest.mark.parametrize("P,pre", [(3, True), (5, True), (5, False)])
def test_edits_reach_both_directions(P, pre, bits):
    """Edits of the values and of the transposed values, before and after the plans hold the long rows' values (from the
    second unchanged pass on), with no plan made anew."""
    F = 64
    world = _world(P, F, bits, pre, False)
    g = torch.Generator(device="cuda").manual_seed(3)
    x, grad = (torch.randn(N, F, generator=g, device="cuda") for _ in range(2))
    before = _same(world, x, grad, bits, pre)
    products = dict(world._stacked.products)
    for passes in (1, 3):
        for _ in range(passes):
            before = _same(world, x, grad, bits, pre)
        for m in _mats(world):
            m.storage.value_T().mul_(5)
        after = _same(world, x, grad, bits, pre)
        assert torch.equal(after[0], before[0]) and not torch.equal(after[1], before[1])
        before = _same(world, x, grad, bits, pre)
        for m in _mats(world):
            m.csr()[2].add_(1)
        after = _same(world, x, grad, bits, pre)
        assert not torch.equal(after[0], before[0]) and torch.equal(after[1], before[1])
    assert all(world._stacked.products[k] is p for k, p in products.items())


def _times_two_unseen(world):
    """Edits that no version counter sees."""
    for m in _mats(world):
        m.csr()[2].data.mul_(2)
        m.storage.value_T().data.mul_(2)


def test_unseen_edits():
    """Rows that are no long rows are read from the caller's tensors by every product; the long rows' values follow after
    a rebinding by hand of the partitions' own plans."""
    g = torch.Generator(device="cuda").manual_seed(4)
    x, grad = (torch.randn(N, 64, generator=g, device="cuda") for _ in range(2))
    short = _world(3, 64, 32, True, False)
    for _ in range(3):
        before = _same(short, x, grad, 32, True)
    _times_two_unseen(short)
    after = _same(short, x, grad, 32, True)
    assert not torch.equal(after[0], before[0]) and not torch.equal(after[1], before[1])
    for rebind in ("bind", "unbind"):
        world = _world(5, 64, 32, True, False)
        for _ in range(3):
            before = _same(world, x, grad, 32, True)
        assert any(p._bound is not None for p in world._stacked.products.values())
        _times_two_unseen(world)
        for m in _mats(world):
            for plan, value in ((m.spmm_plan(), m.csr()[2]), (m.spmm_plan_T(), m.storage.value_T())):
                plan.bind_values(value) if rebind == "bind" else plan.unbind_values()
        for _ in range(3):
            after = _same(world, x, grad, 32, True)
            assert not torch.equal(after[0], before[0]) and not torch.equal(after[1], before[1])


@pytest.mark.parametrize("bits", [32, 2])
def test_replays_read_edited_values(bits):
    from super_gnn_amd.aggregator import Aggregator, _world_forward
    world = _world(3, 64, bits, True, False)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(N, 64, generator=g, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.no_grad():
        for _ in range(3):
            Aggregator.apply(world, x, 0, bits, True, True)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        out = Aggregator.apply(world, x, 0, bits, True, True)
    results = []
    for _ in range(4):
        for m in _mats(world):
            m.csr()[2].mul_(1.5)
        x.add_(0.25)
        graph.replay()
        torch.cuda.synchronize()
        with torch.no_grad():
            want = Aggregator.apply(world, x, 0, bits, True, True)
        plain = torch.cat(_world_forward(world, torch.split(x, world.partition_sizes), bits))
        assert torch.equal(out, plain) and torch.equal(want, plain)
        results.append(out.clone())
    assert not torch.equal(results[0], results[1])


def test_a_wrong_number_of_values_is_refused():
    world = _world(3, 64, 32, True, False)
    x = torch.randn(N, 64, device="cuda")
    _both(world, x, x, 32, True)
    a, b = world.graphs[0].local_adj_t, world.graphs[1].local_adj_t   # the total stays what it was
    a._value, b._value = a._value[:-1].contiguous(), torch.cat([b._value, b._value[:1]])
    from super_gnn_amd.aggregator import Aggregator
    with pytest.raises(ValueError, match="entries"):
        Aggregator.apply(world, x, 0, 32, True, True)


@pytest.mark.parametrize("bits", [32, 4])
def test_no_stacking_where_the_parts_take_bands(bits, monkeypatch):
    from super_gnn_amd.supergnn_ops import SpmmPlan
    monkeypatch.setenv("SGNN_SPMM_BAND", "1")
    monkeypatch.setattr(SpmmPlan, "stack", classmethod(lambda cls, plans: pytest.fail("stacked in vain")))
    x = torch.randn(N, 64, generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")
    _same(_world(3, 64, bits, True, False), x, x.flip(0).contiguous(), bits, True)


@pytest.mark.parametrize("error", ["memory", "library", "argument", "thresholds"])
def test_the_parts_run_where_stacking_is_refused(error, monkeypatch):
    from super_gnn_amd import _lib
    from super_gnn_amd.supergnn_ops import SpmmPlan
    world = _world(3, 64, 32, True, False)
    if error == "thresholds":
        m = world.graphs[1].local_adj_t
        m._plan = SpmmPlan(*m.csr()[:2], m.sparse_size(1), long_row_threshold=4)
    else:
        what = {"memory": torch.cuda.OutOfMemoryError, "library": _lib.SgnnError, "argument": ValueError}[error]

        def refuse(cls, plans):
            raise what("no")
        monkeypatch.setattr(SpmmPlan, "stack", classmethod(refuse))
    x = torch.randn(N, 64, generator=torch.Generator(device="cuda").manual_seed(7), device="cuda")
    for _ in range(2):
        _same(world, x, x.flip(0).contiguous(), 32, True)
    outs = world.aggregate(torch.split(x, world.partition_sizes))
    from super_gnn_amd.aggregator import _world_forward
    assert all(torch.equal(a, b) for a, b in zip(outs, _world_forward(world, torch.split(x, world.partition_sizes), 32)))


@pytest.mark.parametrize("bits", [32, 4])
@pytest.mark.parametrize("pre,kind", [(True, "missing"), (True, "empty"), (False, "empty")])
def test_a_partition_without_neighbours(pre, kind, bits):
    """Nothing is exchanged with the last partition: the matrices it holds for that may be missing or have no rows at all."""
    from super_gnn_amd import SparseTensor, synth
    from super_gnn_amd.aggregator import Aggregator, LoopbackWorld, _world_forward
    from super_gnn_amd.data_manager import build_loopback_partitions
    n = N // 3
    rowptr, col = synth.uniform_degree_graph(2 * n, 7, seed=8)
    rowptr = torch.cat([rowptr, rowptr[-1] + torch.arange(1, n + 1)])
    col = torch.cat([col, torch.arange(2 * n, 3 * n, dtype=col.dtype)])   # the last third: self loops alone
    graphs = build_loopback_partitions(rowptr, col, torch.rand(col.numel()), 3, 64, num_bits=bits, is_pre_delay=pre)
    last = graphs[2]
    assert sum(last.comm_splits.send_splits) == sum(last.comm_splits.recv_splits) == 0
    none = torch.zeros(0, dtype=torch.int64, device="cuda")
    empty = SparseTensor(rowptr=torch.zeros(1, dtype=torch.int64, device="cuda"), col=none, value=none.float(), sparse_sizes=(0, 0))
    if pre:
        last.adj_t_pre_post_aggr_to = None if kind == "missing" else empty
        last.adj_t_pre_post_aggr_from = empty
    else:
        last.remote_adj_t = empty
    world = LoopbackWorld(graphs, bits, pre)
    x = torch.randn(N, 64, generator=torch.Generator(device="cuda").manual_seed(8), device="cuda")
    a = x.clone().requires_grad_()
    out = Aggregator.apply(world, a, 0, bits, pre, True)
    out.backward(x)
    assert torch.equal(out, torch.cat(_world_forward(world, torch.split(x, world.partition_sizes), bits)))
    lone = graphs[2].local_adj_t.csr()[2][:, None] * x[2 * n:]
    assert torch.equal(out[2 * n:], lone) and torch.equal(a.grad[2 * n:], lone)


@pytest.mark.parametrize("dtype", [torch.int64, torch.float64])
def test_edge_values_of_other_types(dtype):
    """They are converted for the product, as SPMM_forward does."""
    from super_gnn_amd.aggregator import Aggregator, LoopbackWorld, _world_forward
    world = _world(3, 64, 32, True, False)
    m = world.graphs[1].local_adj_t
    m._value = (m._value * 8).to(dtype)
    x = torch.randn(N, 64, generator=torch.Generator(device="cuda").manual_seed(9), device="cuda")
    out = Aggregator.apply(LoopbackWorld(world.graphs, 32, True), x, 0, 32, True, True)
    assert torch.equal(out, torch.cat(_world_forward(LoopbackWorld(world.graphs, 32, True), torch.split(x, world.partition_sizes), 32)))


@pytest.mark.parametrize("bits", [32, 4])
@pytest.mark.parametrize("bad", [N // 3, -1])
def test_boundary_rows_beyond_the_partition_are_refused(bad, bits):
    """Stacked, such an index would pick a row of another partition."""
    from super_gnn_amd.aggregator import Aggregator
    world = _world(3, 64, bits, False, False)
    x = torch.randn(N, 64, device="cuda")
    Aggregator.apply(world, x, 0, bits, False, True)
    world.graphs[1 if bad < 0 else 0].idx_nodes_send_to_others[0] = bad
    with pytest.raises(IndexError):
        Aggregator.apply(world, x, 0, bits, False, True)


@pytest.mark.parametrize("bits", [32, 4])
@pytest.mark.parametrize("pre", [False, True])
def test_work_ranges(pre, bits):
    """Stacked products leave the work ranges that the partitions' own products leave."""
    from super_gnn_amd.aggregator import Aggregator, _world_backward, _world_forward
    one, other = _world(3, 64, bits, pre, False), _world(3, 64, bits, pre, False)
    x = torch.randn(N, 64, device="cuda", requires_grad=True)
    Aggregator.apply(one, x, 0, bits, pre, True).sum().backward()
    rows = torch.split(x.detach(), other.partition_sizes)
    _world_forward(other, rows, bits)
    _world_backward(other, rows, bits)
    for a, b in zip(_mats(one), _mats(other)):
        for ask in ("get_work_range", "get_work_range_for_transpose"):
            for got, want in zip(getattr(a, ask)(), getattr(b, ask)()):
                assert torch.equal(got, want)


@pytest.mark.parametrize("P,F,separate,stacked", [(2, 64, False, True), (2, 64, True, False), (8, 64, True, True)])
def test_worlds_that_are_stacked(P, F, separate, stacked, monkeypatch):
    """Two partitions that come as tensors of their own are not worth the copies."""
    from super_gnn_amd.aggregator import Aggregator, _world_forward, _worth_stacking
    from super_gnn_amd.supergnn_ops import SpmmPlan
    made, stack = [], SpmmPlan.stack
    monkeypatch.setattr(SpmmPlan, "stack", classmethod(lambda cls, plans: made.append(1) or stack(plans)))
    world = _world(P, F, 32, True, False)
    x = torch.randn(N, F, device="cuda")
    rows = torch.split(x, world.partition_sizes)
    out = torch.cat(world.aggregate(rows)) if separate else Aggregator.apply(world, x, 0, 32, True, True)
    assert torch.equal(out, torch.cat(_world_forward(world, rows, 32))) and bool(made) == stacked
    # by the floats that a partition's edges gather
    assert _worth_stacking(8, 4_000_000, 128, False) and not _worth_stacking(8, 32_000_000, 128, False)
    assert _worth_stacking(2, 2_000_000, 128, False) and not _worth_stacking(2, 4_000_000, 128, False)
    assert _worth_stacking(8, 4_000_000, 128, True) and not _worth_stacking(8, 8_000_000, 128, True)
