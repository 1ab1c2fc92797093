"""The quantizers' native short cut: it takes plain GPU tensors alone, and answers 0 -- the wrappers' own path, with its staging
and its errors -- for everything else."""
import pytest
import torch


def _args(dev, n=40, F=12, bits=4, wire=False):
    from super_gnn_amd import supergnn_ops as ops
    x = torch.randn(n, F, generator=torch.Generator().manual_seed(n)).to(dev)
    q = torch.zeros((n + 1) // 2, F, dtype=torch.uint8, device=dev)
    p = torch.zeros(n, 2, dtype=torch.bfloat16 if wire else torch.float32, device=dev)
    seg, pseg = (torch.tensor(v, dtype=torch.int32, device=dev) for v in ([0, n], [0, (n + 1) // 2]))
    return ops._direct, [x, q, p, seg, pseg, n, (n + 1) // 2, bits]


def test_takes_nothing_without_a_gpu_and_nothing_that_is_no_tensor():
    direct, args = _args("cpu")
    assert direct.quant_rows(*args) == 0 and direct.dequant_rows(*args) == 0
    assert direct.quant_rows(1, 2, 3, 4, 5, 6, 7, 8) == 0 and direct.quant_rows() == 0
    assert direct.dequant_rows(None, None, None, None, None, "a", 1, 8) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("wire", [False, True])
def test_queues_plain_calls_and_refuses_the_rest(wire):
    direct, args = _args("cuda", wire=wire)
    x, q, p = args[:3]
    before = [t.clone() for t in (x, q, p)]
    tr = torch.randn(12, 40, device="cuda").t()

    class Sub(torch.Tensor):
        pass

    bad = [(0, tr), (0, x.double()), (0, x[:-1]), (0, x.reshape(-1)), (0, x.cpu()), (0, x.as_subclass(Sub)), (1, q[:-1]), (1, q.view(torch.int8)),
           (1, torch.zeros(40, 12, dtype=torch.uint8, device="cuda")[::2]), (2, p[:-1]), (2, p.double()), (2, p.cpu()), (3, args[3].long()),
           (4, args[4][:-1]), (5, 41), (6, 1 << 40), (7, "4")]
    for i, t in bad:
        changed = list(args)
        changed[i] = t
        assert direct.quant_rows(*changed) == 0 and direct.dequant_rows(*changed) == 0, i
    assert all(torch.equal(a, b) for a, b in zip((x, q, p), before))
    assert direct.quant_rows(*args[:7], 3) < 0                       # the library's own refusal comes through as its status
    assert direct.quant_rows(*args) == 1
    back = torch.zeros_like(x)
    assert direct.dequant_rows(back, *args[1:]) == 1
    scale = p.float()[:, 1:]
    assert bool(((back - x).abs() <= scale * 0.5 + (0.02 * x.abs().max() if wire else 1e-5)).all())


@pytest.mark.gpu
def test_runs_on_the_current_stream_and_is_captured():
    from super_gnn_amd import supergnn_ops as ops
    _, (x, q, p, *_) = _args("cuda", n=2000, F=128, bits=8)
    q = torch.zeros(2000, 128, dtype=torch.uint8, device="cuda")
    ops.quantize_tensor(x, q, p, 8)
    want = q.clone()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.quantize_tensor(x, q, p, 8)
    for _ in range(3):
        q.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(q, want)
