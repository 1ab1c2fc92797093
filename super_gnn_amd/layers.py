"""GraphSAGE layer and model over the loop-back partitions: the arithmetic of the reference's
``DistSAGEConvGrad.forward`` (super_gnn/layers/sageconv.py:62-89: aggregate, divide by the in-degree,
``lin_neigh(agg) + lin_self(x) + bias``) and of ``DistSAGE.forward`` (examples/graphsage/sage.py:176-211:
conv, dropout, norm, relu per hidden layer, log_softmax at the end), with every partition of the
graph processed in this one process and the weights shared between them (what DistributedDataParallel
replication amounts to on one GPU).  The dense products are plain torch (rocBLAS) GEMMs."""
import math
from typing import List, Sequence

import torch
import torch.nn.functional as F
from torch import Tensor
from torch.nn import LayerNorm, Linear, Parameter

from .aggregator import Aggregator, LoopbackWorld
from .supergnn_ops import add_rest_product, column_sum, norm_relu, norm_relu_backward


def _column_sum(g: Tensor) -> Tensor:
    n, c = g.shape
    if 0 < n < 1 << 31 and c % 4 == 0 and c <= 1024 and _plain(g) and g.data_ptr() % 16 == 0:
        return column_sum(g)
    k = 4 // math.gcd(c, 4)
    if k == 1 or n < k or not g.is_contiguous():
        return g.sum(0)
    m = n // k * k
    s = g[:m].view(m // k, k * c).sum(0).view(k, c).sum(0)
    return s + g[m:].sum(0) if m < n else s


_SPLIT_K = 64


def _addressable(t):
    """Whether a kernel may read the tensor by address: a plain one on the current device with memory of its own, which the
    members of a batch of gradients do not have."""
    return type(t) in (Tensor, Parameter) and t.is_cuda and torch._C._has_storage(t) and t.get_device() == torch.cuda.current_device()


def _plain(*tensors):
    """Tensors a kernel may read by address, in a gradient that is not differentiated itself."""
    return not torch.is_grad_enabled() and all(_addressable(t) and t.dtype == torch.float32 and t.is_contiguous() for t in tensors)


def _weight_grad(g: Tensor, a: Tensor) -> Tensor:
    """g^T @ a for tall operands ([rows, out] and [rows, in], rows >> out, in).  The product has only
    out x in outputs, too few tiles to fill 256 CUs, so the row axis is cut into _SPLIT_K slabs that run as one
    batched GEMM and are then added (measured at 306 k rows: 0.67 -> 0.17 ms for 256 x 128, 0.71 -> 0.32 ms for
    256 x 256, 0.78 -> 0.11 ms for 47 x 256)."""
    n = g.shape[0]
    if n < _SPLIT_K * 1024 or not (g.is_contiguous() and a.is_contiguous()):
        return g.t() @ a
    m = n // _SPLIT_K * _SPLIT_K
    w = torch.bmm(g[:m].view(_SPLIT_K, m // _SPLIT_K, -1).transpose(1, 2), a[:m].view(_SPLIT_K, m // _SPLIT_K, -1)).sum(0)
    if m < n:
        if _plain(g, a, w):
            add_rest_product(g[m:], a[m:], w)
        else:
            w.addmm_(g[m:].t(), a[m:])
    return w


class _SageCombine(torch.autograd.Function):
    """``(agg / deg) @ W_neigh^T + x @ W_self^T + bias`` (sageconv.py:83-89) as two GEMMs that accumulate into one
    output, instead of two products and two elementwise additions.  In the backward pass the bias gradient is
    summed through a [rows / 4, 4 * width] view when the width is not a multiple of 4: torch's column sum of
    a tall [rows, 47] matrix takes 2.4 ms per partition on MI355X (scalar loads), the same bytes viewed
    188 wide take the vectorized path."""

    @staticmethod
    def forward(ctx, agg, x, deg, w_neigh, w_self, bias):
        mean = agg / deg if deg is not None else agg
        out = torch.addmm(bias, x, w_self.t()) if bias is not None else x @ w_self.t()
        out.addmm_(mean, w_neigh.t())
        ctx.save_for_backward(mean, x, deg, w_neigh, w_self)
        ctx.has_bias = bias is not None
        return out

    @staticmethod
    def backward(ctx, g):
        mean, x, deg, w_neigh, w_self = ctx.saved_tensors
        g = g.contiguous()
        need = ctx.needs_input_grad
        g_agg = g_x = g_wn = g_ws = g_b = None
        if need[0]:
            g_agg = g @ w_neigh
            if deg is not None:
                g_agg.div_(deg)
        if need[1]:
            g_x = g @ w_self
        if need[3]:
            g_wn = _weight_grad(g, mean)
        if need[4]:
            g_ws = _weight_grad(g, x)
        if ctx.has_bias and need[5]:
            g_b = _column_sum(g)
        return g_agg, g_x, None, g_wn, g_ws, g_b


class _DropoutNormRelu(torch.autograd.Function):
    """relu(layer_norm(dropout(x))) with the norm and the rectifier in one pass forward, and everything in one pass backward.
    The dropout itself is torch's, so that the masks are those of its generator."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps, p):
        dropped, mask = torch.native_dropout(x, p, True) if p > 0 else (x, None)
        signs = torch.empty((x.shape[0], (x.shape[1] + 7) // 8), dtype=torch.uint8, device=x.device)
        y, stats = norm_relu(dropped, weight, bias, eps, signs)
        ctx.save_for_backward(x, mask, stats, signs, weight, bias)
        ctx.eps, ctx.scale = eps, 1.0 / (1.0 - p)
        return y

    @staticmethod
    def backward(ctx, g):
        x, mask, stats, signs, weight, bias = ctx.saved_tensors
        (n, C), real = g.shape, torch.float32
        expected = ((g, real, (n, C)), (x, real, (n, C)), (mask, torch.bool, (n, C)), (stats, real, (n, 2)),
                    (signs, torch.uint8, (n, (C + 7) // 8)), (weight, real, (C,)), (bias, real, (C,)))
        if torch.is_grad_enabled() or not all(t is None or _addressable(t) and t.dtype == kind and t.shape == shape for t, kind, shape in expected):
            return _norm_relu_gradients(g, x, mask, ctx.scale, ctx.eps, stats, signs, weight) + (None, None)
        # contiguous, yet somewhere inside another tensor, as torch.cat hands gradients back, will not do either
        g, x, mask, stats, signs, weight, bias = (t if t is None or t.is_contiguous() and t.data_ptr() % 16 == 0
                                                  else t.clone(memory_format=torch.contiguous_format) for t, _, _ in expected)
        return norm_relu_backward(g, x, mask, ctx.scale, stats, weight, bias, signs) + (None, None)


def _norm_relu_gradients(g, x, mask, scale, eps, stats, signs, weight):
    """norm_relu_backward in torch's operations: for gradients that are differentiated themselves, which go through the rows' mean
    and deviation too, for batches of gradients, and for tensors that hooks on saved tensors hand back as something else."""
    C = weight.numel()
    passed = (signs.unsqueeze(-1) >> torch.arange(8, dtype=torch.uint8, device=signs.device) & 1).flatten(1)[:, :C].bool()
    if mask is not None:
        x = x * mask * scale
    if torch.is_grad_enabled():
        mean, rstd = x.mean(1, keepdim=True), (x.var(1, unbiased=False, keepdim=True) + eps).rsqrt()
    else:
        mean, rstd = stats[:, :1], stats[:, 1:]
    hat = (x - mean) * rstd
    g = torch.where(passed, g, 0.0)
    gh = g * weight
    gx = (gh - gh.mean(1, keepdim=True) - hat * (gh * hat).mean(1, keepdim=True)) * rstd
    if mask is not None:
        gx = gx * mask * scale
    return gx, (g * hat).sum(0), g.sum(0)


_global_hooks = getattr(torch.nn.modules.module, "_has_any_global_hook", lambda: False)
_layer_norm_forward = LayerNorm.forward


def _watched():
    """Whether something sees or transforms the operations that run: autocast, tracing, function and dispatch modes, torch.func,
    forward-mode differentiation."""
    return (torch.is_autocast_enabled() or torch.jit.is_tracing() or torch.compiler.is_compiling() or torch._C._len_torch_function_stack() > 0
            or torch._C._len_torch_dispatch_stack() > 0 or torch._C._are_functorch_transforms_active()
            or torch.autograd.forward_ad._current_level >= 0)


def _fusable(norm, x):
    """Whether the one-pass kernels stand for dropout, ``norm`` and the rectifier: a plain LayerNorm over fp32 rows on the GPU,
    with nothing attached that would see the modules' own calls."""
    if type(norm) is not LayerNorm or type(x) is not Tensor or not _addressable(x) or x.dtype != torch.float32 or x.dim() != 2:
        return False
    n, C = x.shape
    if n == 0 or n >= 1 << 31 or C % 4 or C > 1024 or tuple(norm.normalized_shape) != (C,) or not x.is_contiguous() or x.data_ptr() % 16:
        return False
    for t in (norm.weight, norm.bias):
        if type(t) is not Parameter or t.dtype != torch.float32 or t.device != x.device or not t.is_contiguous() or t.data_ptr() % 16:
            return False
    if norm._forward_hooks or norm._forward_pre_hooks or norm._backward_hooks or norm._backward_pre_hooks or _global_hooks():
        return False
    if "forward" in norm.__dict__ or LayerNorm.forward is not _layer_norm_forward:   # another forward put in its place
        return False
    return not _watched()


def _dropout_norm_relu(x, norm, p, training):
    """The stretch between two convolutions (sage.py:186-204)."""
    if norm is not None and 0 <= p < 1 and _fusable(norm, x):
        return _DropoutNormRelu.apply(x, norm.weight, norm.bias, norm.eps, p if training else 0.0)
    x = F.dropout(x, p=p, training=training)
    if norm is not None:
        x = norm(x)
    return F.relu(x)


class LoopbackSAGEConv(torch.nn.Module):
    def __init__(self, in_channels: int, out_channels: int, normalize: bool = True, bias: bool = True):
        super().__init__()
        self.in_channels, self.out_channels, self.normalize = in_channels, out_channels, normalize
        self.lin_neigh = Linear(in_channels, out_channels, bias=False)
        self.lin_self = Linear(in_channels, out_channels, bias=False)
        if bias:
            self.bias = Parameter(torch.zeros(out_channels))
        else:
            self.register_parameter("bias", None)

    def reset_parameters(self):
        gain = torch.nn.init.calculate_gain("relu")
        torch.nn.init.xavier_uniform_(self.lin_neigh.weight, gain=gain)
        torch.nn.init.xavier_uniform_(self.lin_self.weight, gain=gain)

    def forward(self, world: LoopbackWorld, feats: Sequence[Tensor]) -> List[Tensor]:
        aggregated = world.aggregate(feats)
        outs = []
        for g, agg, x in zip(world.graphs, aggregated, feats):
            outs.append(_SageCombine.apply(agg, x, g.in_degrees if self.normalize else None,
                                           self.lin_neigh.weight, self.lin_self.weight, self.bias))
        return outs


class LoopbackSAGE(torch.nn.Module):
    def __init__(self, in_channels, hidden_channels, out_channels, num_layers=3, dropout=0.5, norm_type="LayerNorm"):
        super().__init__()
        dims = [in_channels] + [hidden_channels] * (num_layers - 1) + [out_channels]
        self.convs = torch.nn.ModuleList(LoopbackSAGEConv(a, b) for a, b in zip(dims[:-1], dims[1:]))
        self.norms = torch.nn.ModuleList(LayerNorm(hidden_channels) for _ in range(num_layers - 1)) \
            if norm_type == "LayerNorm" else None
        self.dropout = dropout

    def reset_parameters(self):
        for conv in self.convs:
            conv.reset_parameters()
        if self.norms is not None:
            for norm in self.norms:
                norm.reset_parameters()

    def forward(self, world: LoopbackWorld, feats: Sequence[Tensor]) -> List[Tensor]:
        for i, conv in enumerate(self.convs[:-1]):
            norm = None if self.norms is None else self.norms[i]
            feats = [F.dropout(x, p=self.dropout, training=self.training) for x in conv(world, feats)]   # the generator's order
            feats = [_dropout_norm_relu(x, norm, 0.0, False) for x in feats]
        feats = self.convs[-1](world, feats)
        return [F.log_softmax(x, dim=1) for x in feats]


class DistSAGEConvGrad(torch.nn.Module):
    """The reference's layer with the reference's constructor and call signatures
    (super_gnn/layers/sageconv.py:15-89): ``conv(graph, local_nodes_feat, layer)`` aggregates through
    ``Aggregator.apply(graph, feat, layer, num_bits, is_pre_delay, self.training)``, divides by
    ``graph.in_degrees`` and returns ``lin_neigh(agg) + lin_self(feat) + bias``.  ``graph`` is whatever
    ``Aggregator`` accepts: a partition that is the whole graph, or a LoopbackWorld of P partitions with the
    node features of all of them stacked in partition order."""

    def __init__(self, in_channels: int, out_channels: int, num_bits: int, is_pre_delay: bool,
                 add_self_loops: bool = False, normalize: bool = True, bias: bool = True, **kwargs):
        super().__init__()
        self.in_channels, self.out_channels = in_channels, out_channels
        self.add_self_loops, self.normalize = add_self_loops, normalize
        self.num_bits, self.is_pre_delay = num_bits, is_pre_delay
        self.lin_neigh = Linear(in_channels, out_channels, bias=False)
        self.lin_self = Linear(in_channels, out_channels, bias=False)
        if bias:
            self.bias = Parameter(torch.zeros(out_channels))
        else:
            self.register_parameter("bias", None)

    def reset_parameters(self):
        gain = torch.nn.init.calculate_gain("relu")
        torch.nn.init.xavier_uniform_(self.lin_neigh.weight, gain=gain)
        torch.nn.init.xavier_uniform_(self.lin_self.weight, gain=gain)

    def propagate(self, graph, local_nodes_feat, layer):
        return Aggregator.apply(graph, local_nodes_feat, layer, self.num_bits, self.is_pre_delay, self.training)

    def forward(self, graph, local_nodes_feat, layer) -> Tensor:
        agg = self.propagate(graph, local_nodes_feat, layer)
        deg = graph.in_degrees.reshape(-1, 1) if self.normalize else None
        return _SageCombine.apply(agg, local_nodes_feat, deg, self.lin_neigh.weight, self.lin_self.weight, self.bias)


class DistSAGE(torch.nn.Module):
    """The model of the reference's training script with its constructor and call signatures
    (examples/graphsage/sage.py:127-211; LayerNorm or no norm, no label augmentation)."""

    def __init__(self, in_channels, hidden_channels, out_channels, num_layers=3, dropout=0.5, num_bits=32,
                 is_pre_delay=False, norm_type="LayerNorm", is_label_augment=False):
        super().__init__()
        if is_label_augment:
            raise NotImplementedError("label augmentation (MaskLabel) is outside the aggregation hot path")
        if norm_type not in (None, "LayerNorm"):
            raise NotImplementedError("only LayerNorm (the reference's default) or no normalisation")
        dims = [in_channels] + [hidden_channels] * (num_layers - 1) + [out_channels]
        self.convs = torch.nn.ModuleList(DistSAGEConvGrad(a, b, num_bits, is_pre_delay) for a, b in zip(dims[:-1], dims[1:]))
        self.norms = torch.nn.ModuleList(LayerNorm(hidden_channels) for _ in range(num_layers - 1)) if norm_type else None
        self.dropout, self.norm_type = dropout, norm_type

    def reset_parameters(self):
        for conv in self.convs:
            conv.reset_parameters()
        if self.norms is not None:
            for norm in self.norms:
                norm.reset_parameters()

    def forward(self, graph, nodes_feats, labels=None, label_mask=None):
        for i, conv in enumerate(self.convs[:-1]):
            nodes_feats = conv(graph, nodes_feats, i)
            nodes_feats = _dropout_norm_relu(nodes_feats, None if self.norms is None else self.norms[i], self.dropout, self.training)
        nodes_feats = self.convs[-1](graph, nodes_feats, len(self.convs) - 1)
        return F.log_softmax(nodes_feats, dim=1)
