"""The work a user of this package has it do, as measurable cases: neighbour aggregation (CSR SpMM, forward and
backward), boundary-row quantization in both directions, the fused product over packed rows, one aggregation layer
over loop-back partitions, and one GraphSAGE training step.

Graph and feature sizes are those of this repository's benchmark, tests and training configurations (feature widths
100, 123, 128, 256, 602; 10 k to 2.45 M nodes), or generic ones between them."""
import torch

from super_gnn_amd import (Quantizer_for_all_procs, QuantizerForPureBits, SparseTensor, SPMM_backward, SPMM_forward,
                           SPMM_forward_quantized, synth)
from super_gnn_amd.aggregator import Aggregator, LoopbackWorld
from super_gnn_amd.data_manager import build_loopback_partitions
from super_gnn_amd.layers import DistSAGE

DEVICE = "cuda"


def listed():
    return [
        # A layer of a small graph whose operands live in the caches: what counts is the latency of the call.
        {"name": "spmm_small", "op": "spmm", "graph": "uniform", "nodes": 10_000, "degree": 16, "F": 128,
         "backward": False, "accumulate": False},
        # The gradient of a mid-sized power-law graph's aggregation, at a width that is not a power of two.
        {"name": "spmm_backward", "op": "spmm", "graph": "rmat", "nodes": 200_000, "und_edges": 2_000_000, "F": 100,
         "backward": True, "accumulate": False},
        # The headline product: 2.45 M nodes, 62 M stored edges, GCN weights, accumulated onto out.
        {"name": "spmm_powerlaw", "op": "spmm", "graph": "rmat", "nodes": 2_450_000, "und_edges": 31_000_000, "F": 128,
         "backward": False, "accumulate": True},
        # A dense-degree community graph with wide rows that start on 8-byte boundaries only.
        {"name": "spmm_community", "op": "spmm", "graph": "sbm", "nodes": 233_000, "blocks": 50, "p_in": 0.03048, "F": 602,
         "backward": False, "accumulate": False},
        # Boundary rows of the small graph: one peer, int8.
        {"name": "quant_small", "op": "quantize", "rows": 2_000, "F": 128, "bits": 8, "peers": 1, "gather": False, "wire": False},
        # Boundary rows picked out of the feature matrix for eight peers, (zero_point, scale) in the wire's bf16.
        {"name": "quant_boundary", "op": "quantize", "rows": 500_000, "F": 100, "bits": 4, "peers": 8, "gather": True, "wire": True},
        # The large quantize+pack block.
        {"name": "quant_large", "op": "quantize", "rows": 1_000_000, "F": 256, "bits": 2, "peers": 1, "gather": False, "wire": False},
        # Many short ragged segments of an odd width.
        {"name": "dequant_ragged", "op": "dequantize", "rows": 4_333, "F": 123, "bits": 8, "peers": 256, "wire": False},
        # A large received block of wide rows.
        {"name": "dequant_large", "op": "dequantize", "rows": 425_000, "F": 602, "bits": 4, "peers": 8, "wire": False},
        # Remote rows arrive packed and are accumulated straight onto out.
        {"name": "fused_remote", "op": "fused", "nodes": 1_000_000, "columns": 250_000, "edges": 10_000_000, "F": 128, "bits": 2,
         "peers": 8, "wire": False},
        # One aggregation layer, forward and backward, over eight partitions in pre/post-aggregation mode.
        {"name": "aggregate_layer", "op": "aggregate", "nodes": 200_000, "und_edges": 2_000_000, "F": 128, "bits": 2, "peers": 8,
         "pre": True, "wire": True},
        # One training step of the three-layer model over four partitions that exchange boundary rows as int8.
        {"name": "train_step", "op": "train", "nodes": 150_000, "und_edges": 1_200_000, "F": 100, "hidden": 256, "classes": 47,
         "bits": 8, "peers": 4, "pre": False, "wire": True},
    ]


_WIDTHS = (16, 32, 50, 64, 64, 100, 100, 123, 128, 128, 128, 200, 256, 256, 300, 500, 602, 602, 768, 1024)


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def _width(rng, even=False):
    F = rng.choice(_WIDTHS) if rng.random() < 0.7 else _log(rng, 8, 1024)
    return F + F % 2 if even else F


def draw(rng):
    op = rng.choice(("spmm", "spmm", "spmm", "quantize", "quantize", "dequantize", "fused", "aggregate", "train"))
    if op == "spmm":
        case = {"op": op, "F": _width(rng), "backward": rng.random() < 0.5, "accumulate": rng.random() < 0.5}
        kind = rng.choice(("uniform", "rmat", "rmat", "rmat", "sbm"))
        most = 4e9 / case["F"]   # edges: an edge costs F multiply-adds
        if kind == "uniform":
            n = _log(rng, 1_000, 200_000)
            case.update(graph=kind, nodes=n, degree=max(1, int(min(_log(rng, 2, 64), most / n))))
        elif kind == "rmat":
            n = _log(rng, 2_000, 1_000_000)
            case.update(graph=kind, nodes=n, und_edges=int(min(n * _log(rng, 2, 24), most / 2)))
        else:
            n = _log(rng, 10_000, 100_000)
            blocks = rng.randint(4, 20)
            degree = min(_log(rng, 50, 400), most / n)
            case.update(graph=kind, nodes=n, blocks=blocks, p_in=min(0.5, degree * 20 / (n * (1 + 19 / blocks))))
        return case
    if op in ("quantize", "dequantize"):
        F = _width(rng)
        case = {"op": op, "rows": _log(rng, 500, min(2_000_000, 256_000_000 // F)), "F": F, "bits": rng.choice((8, 4, 2)),
                "peers": rng.choice((1, 2, 4, 8, 16, 64)), "wire": rng.random() < 0.5}
        if op == "quantize":
            case["gather"] = rng.random() < 0.4
        return case
    if op == "fused":
        F = _width(rng, even=True)
        n = _log(rng, 5_000, 1_000_000)
        return {"op": op, "nodes": n, "columns": max(100, n // rng.randint(2, 8)), "edges": int(min(n * _log(rng, 2, 20), 2e9 / F)),
                "F": F, "bits": rng.choice((8, 4, 2)), "peers": rng.choice((2, 4, 8)), "wire": rng.random() < 0.5}
    n = _log(rng, 5_000, 200_000)
    case = {"op": op, "nodes": n, "und_edges": n * _log(rng, 4, 12), "F": rng.choice((64, 100, 128, 256)),
            "bits": rng.choice((32, 8, 4, 2)), "peers": rng.choice((1, 2, 4, 8)), "pre": rng.random() < 0.5, "wire": rng.random() < 0.5}
    if op == "train":
        case.update(hidden=rng.choice((64, 128, 256)), classes=rng.choice((7, 40, 47)))
    return case


# ------------------------------------------------------------------------------------------------
# What the user's program has in hand
# ------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _graph(case, seed, device=DEVICE):
    """(rowptr, col, edge values) of the case's graph: GCN weights on power-law graphs, ones elsewhere."""
    kind = case.get("graph", "rmat")
    if kind == "uniform":
        rowptr, col = synth.uniform_degree_graph(case["nodes"], case["degree"], seed=seed, device=device)
    elif kind == "sbm":
        rowptr, col = synth.sbm_graph(case["nodes"], case["blocks"], case["p_in"], case["p_in"] / 20, seed=seed, device=device)
    else:
        rowptr, col = synth.rmat_graph(case["nodes"], case["und_edges"], seed=seed, device=device)
    value = synth.gcn_norm_weights(rowptr, col) if kind == "rmat" else torch.ones(col.numel(), device=device)
    return rowptr, col, value


def _segments(rows, peers):
    """Cumulative row ranges of `peers` unequal segments."""
    share = torch.arange(1, peers + 1, dtype=torch.float64).sqrt()
    ends = (share.cumsum(0) / share.sum() * rows).round().to(torch.int32)
    return torch.cat([torch.zeros(1, dtype=torch.int32), ends])


def _packed_rows(work_range, bits):
    per_byte = 8 // bits
    sizes = work_range[1:] - work_range[:-1]
    return int(((sizes + per_byte - 1) // per_byte).sum())


def _params(case, rows):
    return torch.empty((rows, 2), dtype=torch.bfloat16 if case["wire"] else torch.float32, device=DEVICE)


def _prepare_spmm(case, seed):
    rowptr, col, value = _graph(case, seed)
    n = case["nodes"]
    matrix = SparseTensor(rowptr=rowptr, col=col, value=value, sparse_sizes=(n, n))
    matrix.spmm_plan_T() if case["backward"] else matrix.spmm_plan()
    x = torch.randn(n, case["F"], generator=_generator(seed + 1), device=DEVICE)
    return {"matrix": matrix, "x": x, "out": torch.zeros_like(x)}


def _prepare_quantize(case, seed):
    rows, F, bits = case["rows"], case["F"], case["bits"]
    work_range = _segments(rows, case["peers"])
    state = {"work_range": work_range, "quantizer": Quantizer_for_all_procs(case["peers"], bits), "row_index": None,
             "data": torch.empty((_packed_rows(work_range, bits), F), dtype=torch.uint8, device=DEVICE), "params": _params(case, rows)}
    if case["gather"]:   # two of three nodes are boundary nodes, in ascending order
        n = rows + rows // 2
        state["row_index"] = torch.randperm(n, generator=_generator(seed + 1), device=DEVICE)[:rows].sort().values
    else:
        n = rows
    state["x"] = synth.boundary_features(n, F, seed=seed, device=DEVICE)
    return state


def _prepare_dequantize(case, seed):
    state = _prepare_quantize(dict(case, gather=False), seed)
    _quantize(case, state)
    state["out"] = state.pop("x")
    return state


def _prepare_fused(case, seed):
    n, columns, F, bits = case["nodes"], case["columns"], case["F"], case["bits"]
    g = _generator(seed)
    # rows draw their remote edges with the skew of a power-law degree distribution, columns are uniform
    row = (torch.rand(case["edges"], generator=g, device=DEVICE).pow(3) * n).to(torch.int64)
    row = torch.randperm(n, generator=g, device=DEVICE)[row]
    col = torch.randint(0, columns, (case["edges"],), generator=g, device=DEVICE)
    rowptr, col = synth.csr_from_pairs(row, col, n, columns, dedupe=False)
    matrix = SparseTensor(rowptr=rowptr, col=col, value=torch.ones(col.numel(), device=DEVICE), sparse_sizes=(n, columns))
    matrix.spmm_plan()
    state = _prepare_quantize({"rows": columns, "F": F, "bits": bits, "peers": case["peers"], "gather": False, "wire": case["wire"]}, seed)
    _quantize(case, state)
    del state["x"]
    state.update(matrix=matrix, out=torch.randn(n, F, generator=g, device=DEVICE))
    return state


def _world(case, seed, width):
    rowptr, col, value = _graph(case, seed)
    if case["op"] == "train":
        value = None
    packed = case["bits"] in (2, 4, 8)
    graphs = build_loopback_partitions(rowptr, col, value, case["peers"], width, num_bits=case["bits"], is_pre_delay=case["pre"],
                                       device=DEVICE)
    return LoopbackWorld(graphs, case["bits"], case["pre"], params_wire_dtype=torch.bfloat16 if packed and case["wire"] else None)


def _prepare_aggregate(case, seed):
    g = _generator(seed + 1)
    x = torch.randn(case["nodes"], case["F"], generator=g, device=DEVICE)
    return {"world": _world(case, seed, case["F"]), "x": x.requires_grad_(),
            "grad": torch.randn(case["nodes"], case["F"], generator=g, device=DEVICE)}


def _prepare_train(case, seed):
    g = _generator(seed + 1)
    torch.manual_seed(seed)
    model = DistSAGE(case["F"], case["hidden"], case["classes"], num_layers=3, dropout=0.5, num_bits=case["bits"],
                     is_pre_delay=case["pre"]).to(DEVICE)
    model.reset_parameters()
    model.train()
    return {"world": _world(case, seed, max(case["F"], case["hidden"])), "model": model, "seed": seed,
            "x": torch.randn(case["nodes"], case["F"], generator=g, device=DEVICE),
            "labels": torch.randint(0, case["classes"], (case["nodes"], 1), generator=g, device=DEVICE)}


# ------------------------------------------------------------------------------------------------
# One pass
# ------------------------------------------------------------------------------------------------
def _spmm(case, state):
    product = SPMM_backward if case["backward"] else SPMM_forward
    product(state["matrix"], state["x"], state["out"], accumulate=case["accumulate"])
    return state["out"]


def _quantize(case, state):
    if case["peers"] == 1 and state["row_index"] is None and not case["wire"]:
        QuantizerForPureBits.quantize_fp32_to_intX(state["x"], state["data"], state["params"], case["bits"])
    else:
        state["quantizer"].quantize_fp32_to_intX(state["x"], state["data"], state["params"], state["work_range"],
                                                 row_index=state["row_index"])
    return state["data"], state["params"]


def _dequantize(case, state):
    state["quantizer"].dequantize_intX_to_fp32(state["data"], state["out"], state["params"], state["work_range"])
    return state["out"]


def _fused(case, state):
    SPMM_forward_quantized(state["matrix"], state["data"], state["params"], state["work_range"], case["bits"], state["out"])
    return state["out"]


def _aggregate(case, state):
    x = state["x"]
    x.grad = None
    out = Aggregator.apply(state["world"], x, 0, case["bits"], case["pre"], True)
    out.backward(state["grad"])
    return out, x.grad


def _train(case, state):
    model = state["model"]
    torch.manual_seed(state["seed"])   # the step's dropout masks
    model.zero_grad(set_to_none=True)
    out = model(state["world"], state["x"])
    loss = -out.gather(1, state["labels"]).mean()
    loss.backward()
    return {"log_probabilities": out, "loss": loss, "gradients": [p.grad for p in model.parameters()]}


_PREPARE = {"spmm": _prepare_spmm, "quantize": _prepare_quantize, "dequantize": _prepare_dequantize, "fused": _prepare_fused,
            "aggregate": _prepare_aggregate, "train": _prepare_train}
_RUN = {"spmm": _spmm, "quantize": _quantize, "dequantize": _dequantize, "fused": _fused, "aggregate": _aggregate, "train": _train}


def prepare(case, seed):
    state = _PREPARE[case["op"]](case, int(seed))
    state["case"] = case
    return state


def run(state):
    return _RUN[state["case"]["op"]](state["case"], state)


# ------------------------------------------------------------------------------------------------
# The same in 64 bits
# ------------------------------------------------------------------------------------------------
def _product64(rowptr, col, value, rows, onto=None):
    """sum of value[e] * rows(col[e]) over every row's edges, in slabs of rows that hold about 2 GB of products;
    ``rows`` gives the dense operand's rows of an index vector in float64."""
    counts = rowptr[1:] - rowptr[:-1]
    ends, n = rowptr.cpu(), counts.numel()
    F = rows(col[:1].to(torch.int64)).shape[1]
    out = torch.zeros(n, F, dtype=torch.float64, device=col.device) if onto is None else onto.double()
    first = 0
    while first < n:
        last = int(torch.searchsorted(ends, ends[first] + 256_000_000 // F, right=True)) - 1
        last = min(n, max(last, first + 1))
        a, b = int(ends[first]), int(ends[last])
        terms = rows(col[a:b].to(torch.int64)).mul_(value[a:b].double()[:, None])
        out[first:last] += torch.segment_reduce(terms, "sum", lengths=counts[first:last], unsafe=True)
        first = last
    return out


def _transposed(rowptr, col, value, columns):
    row = torch.repeat_interleave(torch.arange(rowptr.numel() - 1, device=col.device), rowptr[1:] - rowptr[:-1])
    order = torch.argsort(col, stable=True)
    ends = torch.zeros(columns + 1, dtype=torch.int64, device=col.device)
    ends[1:] = torch.bincount(col.to(torch.int64), minlength=columns).cumsum(0)
    return ends, row[order], value[order]


def _decoded(state, bits, wanted):
    """Rows ``wanted`` of the packed block: code * scale + zero_point."""
    per_byte = 8 // bits
    ends = state["work_range"].to(torch.int64)
    sizes = ends[1:] - ends[:-1]
    packed = torch.zeros_like(ends)
    packed[1:] = ((sizes + per_byte - 1) // per_byte).cumsum(0)
    ends, packed = ends.to(wanted.device), packed.to(wanted.device)
    segment = torch.searchsorted(ends, wanted, right=True) - 1
    inside = wanted - ends[segment]
    shift = (per_byte - 1 - inside % per_byte) * bits
    code = (state["data"][packed[segment] + inside // per_byte].to(torch.int64) >> shift[:, None]) & (2 ** bits - 1)
    params = state["params"].double()[wanted]
    return code.double() * params[:, 1:] + params[:, :1]


def _train64(case, seed):
    """The step with fp32 exchange: mean aggregation, two products, dropout, LayerNorm, rectifier."""
    rowptr, col, _ = _graph(case, seed)
    ones = torch.ones(col.numel(), device=DEVICE)
    there, back = (rowptr, col, ones), _transposed(rowptr, col, ones, case["nodes"])
    degree = (rowptr[1:] - rowptr[:-1]).clamp(min=1).double()[:, None]
    state = _prepare_train(case, seed)
    model, x = state["model"].double(), state["x"].double()
    torch.manual_seed(seed)

    class Aggregate(torch.autograd.Function):
        @staticmethod
        def forward(ctx, v):
            return _product64(*there, lambda i: v[i])

        @staticmethod
        def backward(ctx, g):
            return _product64(*back, lambda i: g[i])

    for i, conv in enumerate(model.convs):
        x = (Aggregate.apply(x) / degree) @ conv.lin_neigh.weight.t() + x @ conv.lin_self.weight.t() + conv.bias
        if i + 1 < len(model.convs):
            x = x * torch.nn.functional.dropout(torch.ones(x.shape, device=DEVICE), p=model.dropout)
            x = torch.relu(model.norms[i](x))
    out = torch.log_softmax(x, 1)
    loss = -out.gather(1, state["labels"]).mean()
    loss.backward()
    return {"log_probabilities": out.detach(), "loss": loss.detach(), "gradients": [p.grad for p in model.parameters()]}


def exact(case, seed):
    op, seed = case["op"], int(seed)
    if op == "spmm":
        rowptr, col, value = _graph(case, seed)
        if case["backward"]:
            rowptr, col, value = _transposed(rowptr, col, value, case["nodes"])
        x = torch.randn(case["nodes"], case["F"], generator=_generator(seed + 1), device=DEVICE)
        return _product64(rowptr, col, value, lambda i: x[i].double())   # out is zero before the first pass
    if op == "quantize":   # the packed codes are whole numbers
        state = _prepare_quantize(case, seed)
        x = state["x"] if state["row_index"] is None else state["x"][state["row_index"]]
        low = x.amin(1).double()
        scale = (x.amax(1).double() - low) / (2 ** case["bits"] - 1)
        return None, torch.stack([low, torch.where(scale == 0, 1.0, scale)], 1)
    if op == "dequantize":
        state = _prepare_dequantize(case, seed)
        return _decoded(state, case["bits"], torch.arange(case["rows"], device=DEVICE))
    if op == "fused":
        state = _prepare_fused(case, seed)
        rowptr, col, value = state["matrix"].csr()
        return _product64(rowptr, col, value, lambda i: _decoded(state, case["bits"], i), onto=state["out"])
    if case["bits"] != 32:   # codes that follow from computed rows: a step of one is far more than any rounding
        return None
    if op == "train":
        return _train64(case, seed)
    rowptr, col, value = _graph(case, seed)
    state = _prepare_aggregate(case, seed)
    x, grad = state["x"].detach(), state["grad"]
    return (_product64(rowptr, col, value, lambda i: x[i].double()),
            _product64(*_transposed(rowptr, col, value, case["nodes"]), lambda i: grad[i].double()))


# ------------------------------------------------------------------------------------------------
# Bounds
# ------------------------------------------------------------------------------------------------
def _edges(case):
    kind = case.get("graph", "rmat")
    if kind == "uniform":
        return case["nodes"] * (case["degree"] + 1)
    if kind == "rmat":
        return 2 * case["und_edges"]
    n, inside = case["nodes"], 1 / case["blocks"]
    return int(n * n * case["p_in"] * (inside + (1 - inside) / 20))


def work(case):
    op, F = case["op"], case["F"]
    if op == "spmm":
        n, e = case["nodes"], _edges(case)
        return {"bytes": 4 * n * F * (3 if case["accumulate"] else 2) + 8 * e + 8 * (n + 1), "flops": 2 * e * F}
    if op in ("quantize", "dequantize"):
        rows = case["rows"]
        return {"bytes": rows * (4 * F + F * case["bits"] / 8 + (4 if case["wire"] else 8) + (8 if case.get("gather") else 0)), "flops": 4 * rows * F}
    if op == "fused":
        n, k, e = case["nodes"], case["columns"], case["edges"]
        return {"bytes": 8 * n * F + k * (F * case["bits"] / 8 + (4 if case["wire"] else 8)) + 8 * e + 8 * (n + 1), "flops": 4 * e * F}
    n, e = case["nodes"], _edges(case)
    if op == "aggregate":   # both directions: the rows in, the rows out, the edges
        return {"bytes": 2 * (8 * n * F + 8 * e + 8 * n), "flops": 4 * e * F}
    # Three layers: aggregation forward (and backward, except of the input features), two products per layer and their
    # gradients; every layer's rows are read and written once in each direction.
    H, C = case["hidden"], case["classes"]
    aggregated = F + 2 * H + 2 * H
    products = 2 * 2 * n * (F * H + H * H + H * C)
    return {"bytes": 8 * n * (F + 2 * H + C) * 2 + 5 * 8 * e, "flops": 2 * e * aggregated + 3 * products - 2 * 2 * n * F * H}


def tolerance(case):
    op, bits = case["op"], case["bits"] if "bits" in case else 32
    if op == "quantize":
        return "exact"        # bytes and (zero_point, scale)
    if op == "dequantize":
        return {"rel": 1e-7, "max": 1e-6}    # one rounding of code * scale + zero_point
    if op in ("spmm", "fused"):
        # Against sums in 64 bits: 0.6e-7 ... 0.8e-7 at 10 ... 20 edges per row, 4e-7 (max 3.2e-6) at 490.
        return {"rel": 1.6e-6, "max": 1.3e-5}
    # Both below: four times what half of the inputs one bit further away from zero do to the outputs.  A sum that
    # rounds the other way moves a code of the exchanged rows by one step now and then, which is a large change of
    # a few values (1/3 of a row's range at int2), and in training a rectifier may switch with it.
    if op == "aggregate":
        return {"rel": 1e-6, "max": 3e-5} if bits == 32 else {"rel": 1e-3, "max": {8: 0.3, 4: 0.9, 2: 0.99}[bits]}
    rel, most = {32: (2e-3, 0.06), 8: (5e-3, 0.07), 4: (1.5e-2, 0.13), 2: (3e-2, 0.8)}[bits]
    return {"rel": rel, "max": most}
