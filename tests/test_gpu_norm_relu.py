"""dropout -> LayerNorm -> relu in one pass each way, against torch in float64 on the CPU."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _inputs(n, C, seed):
    g = torch.Generator().manual_seed(seed)
    x, go = torch.randn(n, C, generator=g) * 3 + 1, torch.randn(n, C, generator=g)
    return x, go, torch.randn(C, generator=g), torch.randn(C, generator=g)


# widths either side of every lane group's (32, 64, 128, 256, 512 floats) and ragged ones; row counts either side of two rows in flight
@pytest.mark.parametrize("n,C", [(1, 4), (2, 32), (3, 36), (129, 64), (130, 68), (777, 100), (1000, 128), (511, 132), (40001, 256), (333, 260),
                                 (300, 512), (301, 516), (257, 1024)])
@pytest.mark.parametrize("masked", [False, True])
def test_norm_relu_matches_float64(n, C, masked):
    from super_gnn_amd.supergnn_ops import norm_relu, norm_relu_backward
    x, go, w, b = _inputs(n, C, n + C)
    mask = (torch.rand(n, C, generator=torch.Generator().manual_seed(5)) < 0.5) if masked else None
    scale = 2.0 if masked else 1.0
    xr, wr, br = (t.double().requires_grad_() for t in (x, w, b))
    h = F.layer_norm(xr * mask * scale if masked else xr, (C,), wr, br, 1e-5)
    ref = F.relu(h)
    dev = [t.cuda() for t in (x, go, w, b)]
    dropped = dev[0] * mask.cuda() * scale if masked else dev[0]
    y, stats = norm_relu(dropped, dev[2], dev[3], 1e-5)
    # a row's value: a handful of roundings of mean, deviation, quotient and product, each relative to |h - b| and |b|
    bound = 16 * EPS * ((h - br).abs() + br.abs() + 3 * wr.abs()).detach()
    assert bool(((y.double().cpu() - ref.detach()).abs() <= bound).all())
    # the rectifier's side may differ where h is a rounding away from 0: those elements' gradients are taken out of both
    sure = h.detach().abs() > bound
    ref.backward((go * sure).double())
    gx, gw, gb = norm_relu_backward((go * sure).cuda(), dev[0], None if mask is None else mask.cuda(), scale, stats, dev[2], dev[3])
    rstd = stats[:, 1:].double().cpu()
    terms = (go.abs() * w.abs()).double()
    size = (terms + terms.mean(1, keepdim=True) + xr.detach().abs().amax(1, keepdim=True) * rstd * terms.mean(1, keepdim=True) * 8) * rstd * scale
    assert bool(((gx.double().cpu() - xr.grad).abs() <= 64 * EPS * size + 1e-12).all())
    hat = ((h - br) / wr).detach().abs()
    for got, want, mass in ((gw, wr.grad, (go.abs().double() * hat).sum(0)), (gb, br.grad, go.abs().double().sum(0))):
        assert bool(((got.double().cpu() - want).abs() <= (n ** 0.5 + 32) * EPS * mass + 1e-12).all())


def test_same_masks_and_gradients_as_the_separate_modules():
    from super_gnn_amd import layers
    x, go, w, b = (t.cuda() for t in _inputs(3000, 256, 1))
    norm = torch.nn.LayerNorm(256).cuda()
    with torch.no_grad():
        norm.weight.copy_(w); norm.bias.copy_(b)
    got = []
    for fused in (True, False):
        if not fused:
            norm.register_forward_hook(lambda *a: None)    # something that watches the module: its own call is made
        xs = x.clone().requires_grad_()
        norm.zero_grad()
        torch.manual_seed(3)
        assert layers._fusable(norm, xs) == fused
        y = layers._dropout_norm_relu(xs, norm, 0.5, True)
        y.backward(go)
        got.append((y.detach(), xs.grad, norm.weight.grad.clone(), norm.bias.grad.clone()))
    assert bool(((got[0][0] == 0) == (got[1][0] == 0)).float().mean() > 0.99999)
    for a, c in zip(*got):
        assert torch.allclose(a, c, rtol=1e-4, atol=1e-4 * float(c.abs().max()))


def test_special_values_and_second_derivatives():
    from super_gnn_amd import layers
    norm = torch.nn.LayerNorm(64).cuda()
    x = torch.randn(4, 64, device="cuda")
    x[0, 3], x[1, 5], x[2] = float("nan"), float("inf"), 7.0      # a NaN row, an infinite row, a constant row
    y, ref = layers._dropout_norm_relu(x, norm, 0.0, True), F.relu(F.layer_norm(x, (64,), norm.weight, norm.bias))
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and bool((y[2] == 0).all()) and torch.allclose(y[3], ref[3], atol=1e-6)
    xs = torch.randn(5, 64, device="cuda", requires_grad=True)
    grads = []
    for f in (lambda t: layers._dropout_norm_relu(t, norm, 0.0, True), lambda t: F.relu(F.layer_norm(t, (64,), norm.weight, norm.bias))):
        first, = torch.autograd.grad((f(xs) ** 2).sum(), xs, create_graph=True)
        grads.append(torch.autograd.grad((first ** 2).sum(), xs)[0])
    assert torch.allclose(*grads, rtol=1e-3, atol=1e-4)


@pytest.mark.parametrize("n,C", [(1, 4), (3, 36), (4, 64), (5, 68), (1023, 128), (4097, 256), (150000, 256), (300, 516), (64, 1024)])
def test_column_sum_matches_float64(n, C):
    from super_gnn_amd.supergnn_ops import column_sum
    x = torch.randn(n, C, generator=torch.Generator().manual_seed(n), dtype=torch.float32)
    got, want = column_sum(x.cuda()).double().cpu(), x.double().sum(0)
    # a thread's chain of n / 4096 rows and a tree over the workgroups: well below a sequential sum's n roundings
    assert bool(((got - want).abs() <= (n ** 0.5 + 16) * EPS * x.abs().double().sum(0)).all())


@pytest.mark.parametrize("rows,n_out,n_in", [(0, 8, 8), (1, 1, 1), (15, 64, 65), (16, 63, 64), (17, 47, 256), (48, 256, 256), (63, 130, 100)])
def test_rest_product_matches_float64(rows, n_out, n_in):
    from super_gnn_amd.supergnn_ops import add_rest_product
    g, a, w = (torch.randn(*s, generator=torch.Generator().manual_seed(s[-1])) for s in ((rows, n_out), (rows, n_in), (n_out, n_in)))
    want, mass = w.double() + g.double().t() @ a.double(), w.abs().double() + g.abs().double().t() @ a.abs().double()
    got = w.cuda()
    add_rest_product(g.cuda(), a.cuda(), got)
    assert bool(((got.double().cpu() - want).abs() <= (rows + 1) * EPS * mass).all())


def test_weight_gradient_of_rows_that_slabs_leave_over():
    from super_gnn_amd.layers import _weight_grad
    for n in (65536, 65537, 65599):
        g, a = (torch.randn(n, c, generator=torch.Generator().manual_seed(c)).cuda() for c in (8, 12))
        want = g.double().t() @ a.double()
        bound = 64 * EPS * (g.abs().double().t() @ a.abs().double())
        with torch.no_grad():
            assert bool(((_weight_grad(g, a).double() - want).abs() <= bound).all())
        assert bool(((_weight_grad(g, a).double() - want).abs() <= bound).all())   # as in a gradient that is differentiated


@pytest.mark.parametrize("C", [4, 12, 64, 100, 256, 260, 516, 1024])
def test_rectifier_side_is_the_forward_passs(C):
    """Gradients pass where the output is above 0 and nowhere else, also for elements a rounding away from 0 behind a dropout whose
    factor 1 / (1 - p) may be rounded in more ways than one."""
    from super_gnn_amd import layers
    from super_gnn_amd.supergnn_ops import norm_relu
    norm = torch.nn.LayerNorm(C).cuda()
    g = torch.Generator().manual_seed(C)
    for p in (0.04, 0.09, 0.128, 0.5):
        for seed in range(20):
            x = (torch.randn(1, C, generator=g) * 3 + 1).cuda().requires_grad_()
            torch.manual_seed(seed)
            dropped = F.dropout(x.detach(), p)
            stats = norm_relu(dropped, torch.ones_like(norm.weight), torch.zeros_like(norm.bias), norm.eps)[1]
            with torch.no_grad():   # the norm's output is 0 or one rounding of it
                norm.bias.copy_(torch.nextafter(-(dropped[0] - stats[0, 0]) * stats[0, 1], torch.randn(C, generator=g).sign().cuda() * 1e3))
            norm.zero_grad()
            torch.manual_seed(seed)
            y = layers._dropout_norm_relu(x, norm, p, True)
            y.backward(torch.ones_like(y))
            assert torch.equal(norm.bias.grad != 0, y[0] > 0), (p, seed)


def test_dropped_elements_of_rows_that_are_not_finite():
    """A NaN row and an infinite row behind a dropout: every gradient NaN where the separate modules' is, dropped elements included."""
    from super_gnn_amd import layers
    x = torch.randn(6, 64, generator=torch.Generator().manual_seed(1)).cuda()
    x[0, 3], x[1, 5] = float("nan"), float("inf")
    go = torch.randn(6, 64, generator=torch.Generator().manual_seed(2)).cuda()
    go[4, 7], go[5, 9] = float("inf"), float("nan")
    found = []
    for fused in (True, False):
        norm = torch.nn.LayerNorm(64).cuda()
        if not fused:
            norm.register_forward_hook(lambda *a: None)
        xs = x.clone().requires_grad_()
        torch.manual_seed(4)
        assert layers._fusable(norm, xs) == fused
        y = layers._dropout_norm_relu(xs, norm, 0.5, True)
        y.backward(go)
        found.append((y.detach(), xs.grad, norm.weight.grad, norm.bias.grad))
    for a, b in zip(*found):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))


def test_gradients_that_begin_inside_another_tensor():
    from super_gnn_amd import layers
    norm = torch.nn.LayerNorm(64).cuda()
    x = torch.randn(30, 64, generator=torch.Generator().manual_seed(1)).cuda().requires_grad_()
    go = torch.randn(30 * 64 + 1, generator=torch.Generator().manual_seed(2)).cuda()
    y = layers._dropout_norm_relu(x, norm, 0.0, True)
    torch.cat([x.new_zeros(1), y.reshape(-1)]).backward(go)      # y's part starts at element 1
    got = x.grad.clone(), norm.weight.grad.clone(), norm.bias.grad.clone()
    x.grad = None
    norm.zero_grad()
    y = layers._dropout_norm_relu(x, norm, 0.0, True)
    y.backward(go[1:].clone().view(30, 64))
    assert all(torch.equal(a, b) for a, b in zip(got, (x.grad, norm.weight.grad, norm.bias.grad)))


def _stretch(x, norm, p, fused):
    """The stretch through the one-pass kernels, or as the separate modules with the same masks."""
    from super_gnn_amd import layers
    torch.manual_seed(4)
    if fused:
        assert layers._fusable(norm, x)
        return layers._dropout_norm_relu(x, norm, p, True)
    return F.relu(norm(F.dropout(x, p)))


def _close(a, b):
    return torch.allclose(a, b, rtol=1e-4, atol=1e-5 * float(b.detach().abs().max()))   # a few roundings, and sums over 30 rows


@pytest.mark.parametrize("p", [0.0, 0.5])
def test_rows_that_come_from_the_norms_own_weight(p):
    """A gradient that is differentiated itself, of rows that depend on the weight by another way as well: each way counts once."""
    norm = torch.nn.LayerNorm(64).cuda()
    base, w = torch.randn(30, 64, generator=torch.Generator().manual_seed(1)).cuda(), norm.weight
    with torch.no_grad():
        norm.bias.normal_(generator=torch.Generator("cuda").manual_seed(1))
    found = []
    for fused in (True, False):
        first, = torch.autograd.grad((_stretch(base * w, norm, p, fused) ** 2).sum(), w, create_graph=True)
        second, = torch.autograd.grad((first ** 2).sum(), w)
        found.append((first.detach(), second))
    assert _close(found[0][0], found[1][0]) and torch.allclose(found[0][1], found[1][1], rtol=1e-3, atol=1e-4 * float(found[1][1].abs().max()))


@pytest.mark.parametrize("p", [0.0, 0.5])
def test_hooks_on_saved_tensors_and_batches_of_gradients(p):
    """Hooks may hand saved tensors back in another memory order, on other storage or as another type; a batch of gradients has no
    memory that a kernel could read."""
    norm = torch.nn.LayerNorm(64).cuda()
    x = torch.randn(30, 64, generator=torch.Generator().manual_seed(1)).cuda().requires_grad_()
    go = torch.randn(3, 30, 64, generator=torch.Generator().manual_seed(2)).cuda()
    inputs = (x, norm.weight, norm.bias)
    want = [torch.autograd.grad(_stretch(x, norm, p, False), inputs, g) for g in go]

    def turned(t):
        return t.t().contiguous().t() if t.dim() == 2 else t.clone()

    for pack, unpack in ((lambda t: t, turned), (lambda t: t.cpu(), lambda t: t.cuda()),
                         (lambda t: t.double() if t.is_floating_point() else t, lambda t: t)):
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = _stretch(x, norm, p, True)
        got = torch.autograd.grad(y, inputs, go[0])
        assert all(_close(a.to(b.dtype), b) for a, b in zip(got, want[0]))
    got = torch.autograd.grad(_stretch(x, norm, p, True), inputs, go, is_grads_batched=True)
    for i in range(3):
        assert all(_close(a[i], b) for a, b in zip(got, want[i]))


def test_bias_gradients_of_a_batch():
    from super_gnn_amd.layers import _SageCombine
    gen = torch.Generator().manual_seed(1)
    agg, x, wn, ws, b = (torch.randn(*s, generator=gen).cuda() for s in ((50, 12), (50, 12), (8, 12), (8, 12), (8,)))
    b.requires_grad_()
    go = torch.randn(3, 50, 8, generator=gen).cuda()
    got, = torch.autograd.grad(_SageCombine.apply(agg, x, None, wn, ws, b), b, go, is_grads_batched=True)
    assert _close(got, go.sum(1))


def test_another_forward_is_called(monkeypatch):
    from super_gnn_amd import layers
    norm = torch.nn.LayerNorm(64).cuda()
    x = torch.randn(8, 64, generator=torch.Generator().manual_seed(1)).cuda()
    norm.forward = lambda t: t + 1
    assert torch.equal(layers._dropout_norm_relu(x, norm, 0.5, False), F.relu(x + 1))
    del norm.forward
    monkeypatch.setattr(torch.nn.LayerNorm, "forward", lambda self, t: t + 2)
    assert torch.equal(layers._dropout_norm_relu(x, norm, 0.5, False), F.relu(x + 2))


def test_modes_and_transforms_see_the_operations(monkeypatch):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from super_gnn_amd import layers
    norm = torch.nn.LayerNorm(64).cuda()
    x = torch.randn(3, 8, 64, generator=torch.Generator().manual_seed(1)).cuda()
    plain = [F.relu(norm(t)) for t in x]
    seen = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func.__name__)
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func.__name__)
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatch):
        seen.clear()
        with mode():
            y = layers._dropout_norm_relu(x[0], norm, 0.5, False)
        assert any("layer_norm" in name for name in seen) and torch.equal(y, plain[0])

    def f(t):
        return layers._dropout_norm_relu(t, norm, 0.5, False)

    def ref(t):
        return F.relu(norm(t))

    assert _close(torch.func.vmap(f)(x), torch.stack(plain))
    assert _close(torch.func.grad(lambda t: f(t).sum())(x[0]), torch.func.grad(lambda t: ref(t).sum())(x[0]))
    for a, b in zip(torch.func.jvp(f, (x[0],), (x[1],)), torch.func.jvp(ref, (x[0],), (x[1],))):
        assert _close(a, b)
    with torch.autograd.forward_ad.dual_level():
        tangents = [torch.autograd.forward_ad.unpack_dual(h(torch.autograd.forward_ad.make_dual(x[0], x[1]))).tangent for h in (f, ref)]
    assert _close(*tangents)
    assert layers._fusable(norm, x[0])
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)      # the kernels go to the current device's stream
    assert not layers._fusable(norm, x[0])


def test_column_sums_of_more_rows_than_the_kernel_counts():
    from super_gnn_amd.layers import _column_sum
    n = (1 << 31) + 5
    g = torch.ones(n, 4, device="cuda")
    with torch.no_grad():
        got = _column_sum(g)
    assert bool(((got.double() - n).abs() <= 1e-4 * n).all())
