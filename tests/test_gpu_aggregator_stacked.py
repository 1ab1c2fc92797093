"""The partitions' stacked matrices against the partitions one by one: the same floats, for every exchange format, both
modes, widths with and without the fused remote step, graphs without and with long rows (hubs in some partitions only, so
that regrouped and plain long rows meet in one stacked plan)."""
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
        assert world._stacked is not None
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_edited_values_are_seen():
    world = _world(3, 64, 32, True, False)
    g = torch.Generator(device="cuda").manual_seed(2)
    x, grad = (torch.randn(N, 64, generator=g, device="cuda") for _ in range(2))
    before, _ = _both(world, x, grad, 32, True)
    world.graphs[1].local_adj_t.csr()[2].mul_(2)
    got, want = _both(world, x, grad, 32, True)
    assert torch.equal(got[0], want[0]) and not torch.equal(got[0], before[0])
