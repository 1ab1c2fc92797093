"""The work range a matrix reports is that of its first product, whatever happens to the values or the thread count
between that product and the question (the reference computes and stores it with the first product)."""
import pytest
import torch

from super_gnn_amd import SparseTensor
from super_gnn_amd.ops import spmm_kernel


def _matrix(n=500, device="cpu"):
    g = torch.Generator().manual_seed(0)
    counts = torch.randint(0, 9, (n,), generator=g)
    rowptr = torch.zeros(n + 1, dtype=torch.int64)
    rowptr[1:] = counts.cumsum(0)
    col = torch.randint(0, n, (int(rowptr[-1]),), generator=g)
    value = torch.rand(col.numel(), generator=g)
    return SparseTensor(rowptr=rowptr.to(device), col=col.to(device), value=value.to(device), sparse_sizes=(n, n))


def _check(device):
    for transposed in (False, True):
        m = _matrix(device=device)
        rowptr = m.storage.colptr() if transposed else m.csr()[0]
        value = m.storage.value_T() if transposed else m.csr()[2]
        threads = torch.get_num_threads()
        want = spmm_kernel.distribute_work_for_row(rowptr, value, threads)
        ask = m.get_work_range_for_transpose if transposed else m.get_work_range
        assert ask()[0].numel() == 0
        m.note_use(16, transposed)
        m.note_use(24, transposed)
        value[: value.numel() // 2].mul_(50)
        try:
            torch.set_num_threads(threads + 3)
            rows, cols = ask()
        finally:
            torch.set_num_threads(threads)
        assert torch.equal(rows.cpu(), want) and cols.tolist() == [0, 24]
        assert not torch.equal(spmm_kernel.distribute_work_for_row(rowptr, value, threads), want)
        m.note_use(8, transposed)
        assert ask()[0] is rows and ask()[1].tolist() == [0, 8]


@pytest.mark.parametrize("large", [False, True])
def test_split_of_the_first_product(large, monkeypatch):
    if large:   # the form that keeps the prefix sums
        basis = spmm_kernel.split_basis
        monkeypatch.setattr(spmm_kernel, "split_basis",
                            lambda rowptr, value: (*basis(rowptr, value)[:1], None, spmm_kernel.row_prefix(rowptr, value)))
    _check("cpu")


@pytest.mark.gpu
def test_split_of_the_first_product_on_the_gpu():
    _check("cuda")


def test_a_split_that_was_set_stays():
    m = _matrix()
    rows, cols = torch.tensor([0, 500], dtype=torch.int32), torch.tensor([0, 3], dtype=torch.int32)
    m.set_work_range(rows, cols)
    m.note_use(16)
    assert m.get_work_range()[0] is rows and m.get_work_range()[1].tolist() == [0, 16]


@pytest.mark.parametrize("slab", [1, 7, 64, 10_000])
def test_prefix_in_slabs(slab):
    m = _matrix()
    rowptr, _, value = m.csr()
    value = (value * 16).round()   # whole numbers: every order of the sums is exact
    whole = torch.cat([torch.zeros(1, dtype=torch.float64), value.double().cumsum(0)])[rowptr]
    assert torch.equal(spmm_kernel.row_prefix(rowptr, value, slab), whole)


def test_matrices_and_worlds_saved_before_these_attributes():
    """Objects unpickled from files of an earlier version hold none of the attributes that came later."""
    import copy
    from super_gnn_amd.aggregator import LoopbackWorld
    m = copy.deepcopy(_matrix())
    for name in ("_used_width", "_used_width_T", "_split_basis", "_split_basis_T"):
        m.__dict__.pop(name, None)
    assert m.get_work_range()[0].numel() == 0
    m.note_use(16)
    assert m.get_work_range()[1].tolist() == [0, 16]
    m.note_use(16, transposed=True)
    assert m.get_work_range_for_transpose()[1].tolist() == [0, 16]
    world = LoopbackWorld([], 32, False)
    world.__dict__.pop("_stacked", None)
    assert world._stacked is None
