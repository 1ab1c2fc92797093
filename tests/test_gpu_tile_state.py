"""What the schedules of the SpMM that keep state in the plan may not change: products read the edge values they are given,
whatever ran before on the same plan; captured products keep what they were captured with.  Against the CPU oracle, bit for
bit (every row in CSR order with one fma per edge, under every schedule)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from _util import random_csr

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHORT = (4000, 1500, 80, 602)     # no row of more than 128 edges, and the default rule takes tiles


class _Case:
    """A matrix with its plan, operand and a row sample of the oracle's result."""

    def __init__(self, M, K, deg, F, seed=1, **kw):
        from super_gnn_amd import supergnn_ops as ops
        self.rowptr, self.col, val = random_csr(M, K, deg, seed=seed, **kw)
        self.M, self.K, self.F = M, K, F
        self.plan = ops.SpmmPlan(torch.from_numpy(self.rowptr).to(DEV), torch.from_numpy(self.col).to(DEV), K)
        self.value = torch.from_numpy(val).to(DEV)
        self.x = self.operand(F)
        self.out = torch.empty(M, F, device=DEV)

    def operand(self, F):
        return torch.randn(self.K, F, generator=torch.Generator().manual_seed(F)).to(DEV)

    def product(self, value, x=None, out=None):
        x, out = self.x if x is None else x, self.out if out is None else out
        out.fill_(7.0)
        self.plan.run(value, x, out, accumulate=False)
        return out

    def want(self, value, x=None):
        x = self.x if x is None else x
        rows = 200                                           # from the middle on
        r0 = (self.M - rows) // 2
        lo, hi = self.rowptr[r0], self.rowptr[r0 + rows]
        want = np.zeros((rows, x.shape[1]), np.float32)
        orc.spmm_accumulate(self.rowptr[r0:r0 + rows + 1] - lo, self.col[lo:hi],
                            np.ones(hi - lo, np.float32) if value is None else value[lo:hi].cpu().numpy(), x.cpu().numpy(), want)
        return slice(r0, r0 + rows), want

    def check(self, value, x=None, out=None, what=""):
        rows, want = self.want(value, x)
        equal = np.array_equal((self.out if out is None else out)[rows].cpu().numpy(), want)
        assert equal, what


def test_rows_that_are_not_long_are_read_from_the_callers_array():
    """An edit that no version counter sees, after the plan has bound the values by itself."""
    c = _Case(*SHORT)
    assert c.plan.tiles(c.F)[0] > 0 and c.plan.info()["long_rows"] == 0
    for i in range(3):
        c.product(c.value)
        c.check(c.value, what=i)
    c.value.data.mul_(2)
    c.product(c.value)
    c.check(c.value, what="edited through .data")
    c.value.add_(1)
    c.product(c.value)
    c.check(c.value, what="edited in place")


def _captured(c, value):
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.plan.run(value, c.x, c.out, accumulate=False)
    return graph


@pytest.mark.parametrize("kind", ["short", "long", "short, tiles forced", "bands"])
@pytest.mark.parametrize("bound", [False, True])
def test_replays_and_eager_products_do_not_see_each_others_values(kind, bound, monkeypatch):
    """A captured product reads its own array, edited or not, after eager products with other values, and the eager products
    that follow a replay read theirs."""
    if kind == "short":
        c = _Case(*SHORT)
    else:
        monkeypatch.setenv("SGNN_SPMM_BAND", "1" if kind == "bands" else "2")
        c = _Case(700, 900, 40, 130, **({"hubs": 5, "hub_deg": 600} if kind == "long" else {}))
    for _ in range(3):
        c.product(c.value)
    assert c.plan.tiles(c.F)[1] == (kind != "bands")
    if not bound:
        c.plan.unbind_values()
    graph = _captured(c, c.value)
    other = c.value * 3 + 1
    for i in range(3):
        c.out.fill_(7.0)
        graph.replay()
        c.check(c.value, what=("replay", i))
        eager = torch.empty_like(c.out)
        for j in range(3):                                   # unbound, bound, bound and unchanged
            c.product(other, out=eager)
            c.check(other, out=eager, what=("eager", i, j))
        c.out.fill_(7.0)
        graph.replay()
        c.check(c.value, what=("replay after other values", i))
        c.product(other, out=eager)
        c.check(other, out=eager, what=("eager after a replay", i))
        c.value.mul_(1.5)
        c.out.fill_(7.0)
        graph.replay()
        c.check(c.value, what=("replay of edited values", i))
        torch.cuda.synchronize()


def test_captured_products_keep_the_bound_values_of_long_rows():
    """The row classes read a bound array's long rows from the plan's copy; binding another array gives that one its own."""
    c = _Case(700, 900, 40, 130, hubs=5, hub_deg=600)
    assert c.plan.tiles(c.F) == (0, 0) and c.plan.info()["partitioned"] == 1
    for _ in range(3):
        c.product(c.value)
    first, other = c.out.clone(), c.value * 3 + 1
    c.plan.unbind_values()
    second = c.product(other).clone()
    for _ in range(3):
        c.product(c.value)
    graph = _captured(c, c.value)
    for i in range(3):
        for value, want in ((other, second), (c.value, first)):
            for j in range(3):
                c.product(value)
                assert torch.equal(c.out, want), (i, j)
            c.out.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(c.out, first), i


@pytest.mark.parametrize("kind", ["tiles", "bands", "row classes"])
def test_captured_products_keep_their_buffers(kind, monkeypatch):
    """Wider products later on need a larger workspace, other schedules of the same matrix and larger partial sums; what a
    captured product names stays."""
    monkeypatch.setenv("SGNN_SPMM_BAND", {"tiles": "2", "bands": "1", "row classes": "0"}[kind])
    c = _Case(1500, 1200, 30, 64, hubs=6, hub_deg=700)
    for _ in range(3):
        c.product(c.value)
    first = c.out.clone()
    graph = _captured(c, c.value)
    for F in (80, 96, 112, 130, 602):
        x = c.operand(F)
        wide = torch.empty(c.M, F, device=DEV)
        c.product(c.value, x, wide)
        if kind != "row classes":
            c.check(c.value, x, wide, what=F)
        fresh = [torch.full((1 << 20,), float("nan"), device=DEV) for _ in range(8)]   # whatever has been freed is written over
        c.out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c.out, first), F
        del fresh


def test_widths_in_turn_settle_on_the_streams_there_are(monkeypatch):
    """Four widths that each want another number of rows per wave: three get streams of their own, and from then on nothing
    is built (streams are never given up, so their number says so); a product captured on the first width goes on."""
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    widths = (64, 256, 602, 1024)
    c = _Case(40000, 2500, 30, widths[0])
    assert len({c.plan.tiles(F)[0] for F in widths}) == 4
    c.product(c.value)
    graph = _captured(c, c.value)
    for turn in range(3):
        for F in widths:
            x, out = c.operand(F), torch.empty(c.M, F, device=DEV)
            c.product(c.value, x, out)
            c.check(c.value, x, out, what=(turn, F))
        assert c.plan.tiles(widths[0])[1] == 3, turn
        c.out.fill_(7.0)
        graph.replay()
        c.check(c.value, what=("replay", turn))
        torch.cuda.synchronize()


def test_a_width_that_tiles_do_not_suit_leaves_the_others_theirs():
    """Rows of 300 and 120 edges in turns of 32: 103 rows a wave are even enough, a few are not.  A width that wants few must not
    turn off the streams of one that wants many, for calls that may build nothing either (the row classes they would fall
    back to add long rows up in parts: other bits)."""
    from super_gnn_amd import supergnn_ops as ops
    from super_gnn_amd._lib import check, lib
    M, K, many, few = 24000, 40000, 1024, 320
    rng = np.random.default_rng(5)
    deg = np.where(np.arange(M) // 32 % 2 == 0, 300, 120)
    rowptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    col = rng.integers(0, K, size=rowptr[-1])
    col = col[np.lexsort((col, np.repeat(np.arange(M), deg)))]
    plan = ops.SpmmPlan(torch.from_numpy(rowptr).to(DEV), torch.from_numpy(col).to(DEV), K)
    x = {F: torch.randn(K, F, generator=torch.Generator().manual_seed(F)).to(DEV) for F in (many, few)}
    out = torch.empty(M, many, device=DEV)
    assert plan.tiles(many)[0] == 103

    def noalloc(F, out):
        check(lib.sgnn_spmm_csr_f32_noalloc(plan._h, None, x[F].data_ptr(), out.data_ptr(), F, F, F, 0, None, torch.cuda.current_stream().cuda_stream))

    plan.run(None, x[many], out, accumulate=False)
    first = out.clone()
    lo, hi = rowptr[1000], rowptr[1100]
    want = np.zeros((100, many), np.float32)
    orc.spmm_accumulate(rowptr[1000:1101] - lo, col[lo:hi], np.ones(hi - lo, np.float32), x[many].cpu().numpy(), want)
    equal = np.array_equal(first[1000:1100].cpu().numpy(), want)
    assert equal
    for _ in range(2):
        narrow = torch.empty(M, few, device=DEV)
        plan.run(None, x[few], narrow, accumulate=False)
    assert plan.tiles(many)[0] == 103
    out.fill_(7.0)
    noalloc(many, out)
    assert torch.equal(out, first)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.run(None, x[many], out, accumulate=False)
    for _ in range(3):
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first)


def test_products_of_one_matrix_on_several_streams():
    """Without long rows a plan keeps no state between products that are in flight: operands, values and outputs of two streams
    stay apart, with nothing that orders them, and one stream after the other gets its turn."""
    c = _Case(*SHORT)
    streams = [torch.cuda.Stream() for _ in range(2)]
    sets = []
    for i in range(2):
        x, v = torch.randn(c.K, c.F, device=DEV), torch.rand(c.value.numel(), device=DEV)
        sets.append((x, v, torch.empty_like(c.out)))
    torch.cuda.synchronize()
    for turn in range(20):
        for st, (x, v, out) in zip(streams, sets):
            with torch.cuda.stream(st):
                c.product(v, x, out)
        if turn % 5 == 4:
            torch.cuda.synchronize()
            for x, v, out in sets:
                c.check(v, x, out, what=turn)
                out.zero_()
            streams.reverse()
    assert c.plan.tiles(c.F)[1] == 1


@pytest.mark.parametrize("default_stream", [False, True])
def test_threads_and_captures_beside_each_other(default_stream):
    """Another thread's products, the first of a width among them, neither disturb a capture nor wait for one; a captured
    product that is the plan's first builds nothing."""
    import threading
    c = _Case(*SHORT)
    graph = _captured(c, c.value)
    assert c.plan.tiles(c.F)[1] == 0
    errors, widths = [], (602, 700, 1024)
    sets = {F: (c.operand(F), torch.empty(c.M, F, device=DEV)) for F in widths}
    torch.cuda.synchronize()

    def work(n):
        try:
            with torch.cuda.stream(torch.cuda.default_stream() if default_stream else torch.cuda.Stream()):
                for _ in range(n):
                    for x, out in sets.values():
                        c.plan.run(c.value, x, out, accumulate=False, bind=False)
        except Exception as e:   # noqa: BLE001 (shown below)
            errors.append(e)

    second = torch.cuda.CUDAGraph()
    with torch.cuda.graph(second):
        c.plan.run(c.value, c.x, c.out, accumulate=False, bind=False)
        t = threading.Thread(target=work, args=(2,))
        t.start()
        t.join()
    assert not errors and c.plan.tiles(c.F)[1] > 0
    threads = [threading.Thread(target=work, args=(30,)) for _ in range(3)]
    for t in threads:
        t.start()
    for i in range(30):
        c.out.fill_(7.0)
        (graph, second)[i % 2].replay()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    c.check(c.value)
    for x, out in sets.values():
        c.check(c.value, x, out)


@pytest.mark.parametrize("weighted", [True, False])
def test_other_widths_take_the_streams_there_are_where_nothing_may_be_built(weighted, monkeypatch):
    """Widths that want other numbers of rows, through the non-allocating entry point and captured.  Long rows tell the tile schedule
    from the row classes, which add them up in parts."""
    from super_gnn_amd._lib import check, lib
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    c = _Case(20000, 2500, 30, 1024, hubs=400, hub_deg=1500)
    value = c.value if weighted else None
    hub = int(np.argmax(np.diff(c.rowptr) > 1000))
    c.product(value)
    c.check(value)
    assert c.plan.tiles(c.F)[1] == 1

    def hubs_in_one_chain(x, out):
        lo, hi = c.rowptr[hub], c.rowptr[hub + 1]
        want = np.zeros((1, x.shape[1]), np.float32)
        orc.spmm_accumulate(np.array([0, hi - lo]), c.col[lo:hi], np.ones(hi - lo, np.float32) if value is None else value[lo:hi].cpu().numpy(),
                            x.cpu().numpy(), want)
        return np.array_equal(out[hub].cpu().numpy(), want[0])

    for F in (64, 256, 602):
        x, out = c.operand(F), torch.full((c.M, F), 7.0, device=DEV)
        assert c.plan.tiles(F)[0] != c.plan.tiles(c.F)[0]
        args = (c.plan._h, None if value is None else value.data_ptr(), x.data_ptr(), out.data_ptr(), F, F, F, 0, None)
        check(lib.sgnn_spmm_csr_f32_noalloc(*args, torch.cuda.current_stream().cuda_stream))
        c.check(value, x, out, what=F)
        assert hubs_in_one_chain(x, out), F
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            check(lib.sgnn_spmm_csr_f32(*args, torch.cuda.current_stream().cuda_stream))
        for _ in range(3):
            x.mul_(1.5)
            out.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            c.check(value, x, out, what=F)
            assert hubs_in_one_chain(x, out), F
    assert c.plan.tiles(c.F)[1] == 1


@pytest.mark.parametrize("kind", ["short", "long"])
def test_a_product_captured_behind_a_rebinding(kind, monkeypatch):
    """An edit that the version counter sees, between the products that bound the values and the captured one."""
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    c = _Case(700, 900, 40, 130, **({"hubs": 5, "hub_deg": 600} if kind == "long" else {}))
    for _ in range(3):
        c.product(c.value)
    c.value.add_(1)
    graph = _captured(c, c.value)
    for i in range(3):
        c.out.fill_(7.0)
        graph.replay()
        c.check(c.value, what=("replay", i))
        c.product(c.value)
        c.check(c.value, what=("eager", i))
        torch.cuda.synchronize()


@pytest.mark.parametrize("weighted", [True, False])
def test_row_blocks_under_the_tile_schedule(weighted, monkeypatch):
    """Blocks share one restaged operand, and each has its own streams and its own part of the values."""
    monkeypatch.setenv("SGNN_SPMM_BAND", "2")
    whole = _Case(3000, 2600, 35, 130, hubs=3, hub_deg=800)
    monkeypatch.setenv("SGNN_SPMM_PART_EDGES", str(int(whole.rowptr[-1]) // 5))
    blocks = _Case(3000, 2600, 35, 130, hubs=3, hub_deg=800)
    monkeypatch.delenv("SGNN_SPMM_PART_EDGES")
    value = whole.value if weighted else None
    for F in (130, 64, 200, 130):
        x, a, b = whole.operand(F), torch.empty(3000, F, device=DEV), torch.empty(3000, F, device=DEV)
        for _ in range(3):
            whole.product(value, x, a)
            blocks.product(value, x, b)
            whole.check(value, x, a, what=F)
            assert torch.equal(a, b), F
    assert blocks.plan.tiles(130)[1] > 0


def test_row_blocks_of_which_one_takes_tiles_and_one_bands():
    """By the default rule: a block of even rows streams tiles, one whose rows of 400 and 20 edges lie in runs of 300 does not.  The
    two layouts of the restaged operand are told apart within one product."""
    from super_gnn_amd import supergnn_ops as ops
    M, K, F = 24000, 40000, 602
    rng = np.random.default_rng(6)
    deg = np.full(M, 210)
    deg[M // 2:] = np.where(np.arange(M // 2) // 300 % 2 == 0, 400, 20)
    rowptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    col = rng.integers(0, K, size=rowptr[-1])
    col = col[np.lexsort((col, np.repeat(np.arange(M), deg)))]
    rp, cl, x = torch.from_numpy(rowptr).to(DEV), torch.from_numpy(col).to(DEV), torch.randn(K, F, generator=torch.Generator().manual_seed(1))
    with pytest.MonkeyPatch.context() as m:
        m.setenv("SGNN_SPMM_PART_EDGES", str(int(rowptr[M // 2])))
        plan = ops.SpmmPlan(rp, cl, K)
    halves = [ops.SpmmPlan(rp[a:a + M // 2 + 1] - rp[a], cl[rp[a]:rp[a + M // 2]].clone(), K) for a in (0, M // 2)]
    assert [h.tiles(F)[0] > 0 for h in halves] == [True, False] and all(h.schedule(F)["band"] == 1 for h in halves)
    xd, out = x.to(DEV), torch.empty(M, F, device=DEV)
    for value in (None, torch.rand(col.size, generator=torch.Generator().manual_seed(2))):
        for _ in range(3):
            out.fill_(7.0)
            plan.run(None if value is None else value.to(DEV), xd, out, accumulate=False)
            for r0 in (5000, 17900):
                lo, hi = rowptr[r0], rowptr[r0 + 100]
                want = np.zeros((100, F), np.float32)
                orc.spmm_accumulate(rowptr[r0:r0 + 101] - lo, col[lo:hi], np.ones(hi - lo, np.float32) if value is None else value[lo:hi].numpy(),
                                    x.numpy(), want)
                equal = np.array_equal(out[r0:r0 + 100].cpu().numpy(), want)
                assert equal, r0
