"""SpMM façade with the reference's names and signatures (super_gnn/ops/spmm_kernel.py:46-91).

``SPMM_forward(src, other, out)``  : out += A @ other          (result in ``out``, returns None)
``SPMM_backward(src, other, out)`` : out += A^T @ other

The reference computes an nnz-balanced OpenMP row split on first use and caches it on the matrix
(spmm_kernel.py:49-58); here the object that matters is the GPU schedule (SpmmPlan), cached the same
way.  The row split of a matrix is that of its first product, worked out when ``get_work_range()`` is
called: callers see what the reference would have put there."""
import torch

from ..supergnn_ops import quant_segments, spmm


def distribute_work_for_row(rowptr: torch.Tensor, value: torch.Tensor, num_threads_on_row: int) -> torch.Tensor:
    """Greedy contiguous row split balanced by the per-row sum of ``value``: a range is closed at the
    first row whose addition lifts the running sum above total // threads, and that row opens the
    next range (super_gnn/ops/spmm_kernel.py:8-29).  The reference walks all rows in a Python loop;
    this finds each cut with one binary search over the prefix sums.  Kept for interface parity: the
    GPU kernels balance work through the SpMM plan instead and do not consume the split."""
    if value is None or value.numel() == 0:
        return _row_cuts(None, rowptr.numel() - 1, num_threads_on_row)
    prefix = row_prefix(rowptr.detach().cpu(), value.detach().cpu(), value.numel())
    return _row_cuts(prefix, rowptr.numel() - 1, num_threads_on_row)


def row_prefix(rowptr, value, slab=1 << 24):
    """Sum of the first i rows' values in float64, for every i, where the tensors are; edges in slabs, so that the running
    sums of a large matrix take 256 MB."""
    prefix = torch.zeros(rowptr.numel(), dtype=torch.float64, device=rowptr.device)
    for first in range(0, value.numel(), slab):
        part = value[first:first + slab].to(torch.float64).cumsum(0)
        part = torch.cat([part.new_zeros(1), part])
        prefix += part[(rowptr - first).clamp_(0, part.numel() - 1)]
    return prefix


def _row_cuts(prefix, num_rows, num_threads_on_row):
    row_splits = torch.full((num_threads_on_row + 1,), num_rows, dtype=torch.int32)
    row_splits[0] = 0
    if num_rows == 0 or prefix is None:
        return row_splits
    target = float(torch.div(prefix[-1], num_threads_on_row, rounding_mode="floor"))
    start_sum, first_candidate = 0.0, 0                   # sum before the open range; earliest row that may close it
    for t in range(1, num_threads_on_row + 1):
        k = int(torch.searchsorted(prefix, torch.tensor(start_sum + target, dtype=torch.float64), right=True))
        cut = max(k - 1, first_candidate)                 # first row i with prefix[i+1] - start_sum > target
        if cut >= num_rows:
            break
        row_splits[t] = cut
        start_sum, first_candidate = float(prefix[cut]), cut + 1
    row_splits[-1] = num_rows
    return row_splits


def disribute_work_for_col(other: torch.Tensor, num_threads_on_col: int) -> torch.Tensor:
    """Even split of the feature axis (super_gnn/ops/spmm_kernel.py:31-44; the misspelt name is the
    reference's)."""
    return _col_splits(other.shape[-1], num_threads_on_col)


def split_basis(rowptr, value):
    """What a row split depends on, as it is now: the thread count and the values.  It is taken at a matrix's first product; the
    split itself, which walks the rows on the CPU (235 ms of 2.45 M rows), waits until it is asked for.  Up to 2^24 edges the
    values are copied (10 us); beyond that the rows' prefix sums are kept instead, 8 bytes per row."""
    if value is not None and value.numel():
        value = value.detach()
        if value.numel() > 1 << 24:
            return torch.get_num_threads(), None, row_prefix(rowptr, value, 1 << 24 if value.is_cuda else value.numel())
        value = value.clone()
    return torch.get_num_threads(), value, None


def work_range(row_splits, basis, rowptr, width):
    """(row_splits, col_splits) as a product of this width leaves them; an existing row split is kept."""
    if row_splits.size(0) == 0:
        threads, value, prefix = basis
        if prefix is not None:
            row_splits = _row_cuts(prefix.cpu(), rowptr.numel() - 1, threads)
        else:
            row_splits = distribute_work_for_row(rowptr, value, threads)
    return row_splits, _col_splits(width, 1)


def _col_splits(num_cols, num_threads_on_col):
    target = num_cols // num_threads_on_col
    col_splits = torch.full((num_threads_on_col + 1,), num_cols, dtype=torch.int32)
    for i in range(num_threads_on_col):
        col_splits[i] = i * target
    col_splits[-1] = num_cols
    return col_splits


def SPMM_forward(src, other: torch.Tensor, out: torch.Tensor, accumulate=None) -> None:
    """``accumulate=None`` follows the reference (out += A @ other except on its overwrite branch);
    ``False`` writes out = A @ other, which equals zero-filling out and accumulating, bit for bit,
    without the fill and the read-back."""
    rowptr, col, value = src.csr()
    src.note_use(other.shape[-1])   # the work range is computed when asked for (the tensors alone took 6 us of every call)
    if value is not None:
        value = value.to(other.dtype)
    sparse_row = rowptr.shape[0] - 1
    spmm(rowptr, col, value, other, out, sparse_row, plan=src.spmm_plan(), accumulate=accumulate)
    return None


def SPMM_backward(src, other: torch.Tensor, out: torch.Tensor, accumulate=None) -> None:
    colptr = src.storage.colptr()
    row_T = src.storage.row_T()
    value_T = src.storage.value_T()
    src.note_use(other.shape[-1], transposed=True)
    if value_T is not None:
        value_T = value_T.to(other.dtype)
    sparse_row = colptr.shape[0] - 1
    return spmm(colptr, row_T, value_T, other, out, sparse_row, plan=src.spmm_plan_T(), accumulate=accumulate)


def SPMM_forward_quantized(src, data_int8: torch.Tensor, quantized_params: torch.Tensor,
                           work_range_per_proc: torch.Tensor, num_bits: int, out: torch.Tensor) -> None:
    """out += A @ dequantize(data_int8), the remote / post-aggregation step of the forward pass with
    the boundary rows still packed: replaces ``Quantizer_for_all_procs.dequantize_intX_to_fp32(...)``
    followed by ``SPMM_forward(remote_adj_t, recv_buf, out)`` (super_gnn/aggregator.py:72-93) and
    gives the same floats, without materialising ``recv_buf``."""
    _, _, value = src.csr()
    if value is not None:
        value = value.to(torch.float32)
    segs = quant_segments(work_range_per_proc, num_bits)
    src.spmm_plan().run_quantized(value, data_int8, quantized_params, segs, num_bits, out, accumulate=True)
    return None


def SPMM_backward_quantized(src, data_int8: torch.Tensor, quantized_params: torch.Tensor,
                            work_range_per_proc: torch.Tensor, num_bits: int, out: torch.Tensor) -> None:
    """out += A^T @ dequantize(data_int8): the last step of the backward pass in pre/post-aggregation
    mode with the returned gradient rows still packed; replaces ``dequantize_intX_to_fp32(...)``
    followed by ``SPMM_backward(adj_t_pre_post_aggr_to, send_buf, local_grad)``
    (super_gnn/aggregator.py:159-171) and gives the same floats."""
    value_T = src.storage.value_T()
    if value_T is not None:
        value_T = value_T.to(torch.float32)
    segs = quant_segments(work_range_per_proc, num_bits)
    src.spmm_plan_T().run_quantized(value_T, data_int8, quantized_params, segs, num_bits, out, accumulate=True)
    return None
