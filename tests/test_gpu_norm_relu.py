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
