"""Split-K accumulator words of captured graphs: a capture takes words that are zero already, so the
graph holds no zero fill; without such words, or for more of them than a share, it records one."""
import pytest
import torch

from tests.helpers import make_linear_problem, to_gpu, workspace_for

pytestmark = pytest.mark.gpu


def _call(m, k, n, seed, gpu):
    from uniql_amd import ops
    p = make_linear_problem(m, k, n, seed=seed)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    return lambda: ops.w4a16_gemm_ex(x, b, s, ws, m, n, k)


@pytest.mark.parametrize("room", ["plenty", "one share", "none"])
def test_captures_take_words_of_the_reserve(gpu, monkeypatch, room):
    from uniql_amd import ops
    cleared = []
    lib = ops._capi.load()
    clear = lib.uniql_clear
    monkeypatch.setattr(lib, "uniql_clear", lambda *a: (cleared.append(a[1]), clear(*a))[1])
    first, second = _call(1, 4096, 512, 11, gpu), _call(8, 2048, 1024, 12, gpu)
    share = 8 * 1024  # words of the larger call
    ops.reset_accumulators()
    monkeypatch.setattr(ops, "_RESERVE_WORDS", {"plenty": ops._RESERVE_WORDS, "one share": share + 512, "none": 0}[room])
    want = first().clone(), second().clone()
    graphs, outs = [], []
    for _ in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            outs.append((first(), second()))
        graphs.append(g)
    taken = [b for b in ops._accum_in_capture.values()] + ops._accum_retired
    spans = sorted((b.data_ptr(), b.data_ptr() + 8 * b.numel()) for b in taken)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])), "captures share words"
    assert len(cleared) == {"plenty": 0, "one share": 1, "none": 2}[room]
    for _ in range(3):
        for g, o in reversed(list(zip(graphs, outs))):
            for y in o:
                y.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(o[0], want[0]) and torch.equal(o[1], want[1])
        assert torch.equal(first(), want[0])
    del graphs
    assert all(int(b.count_nonzero()) == 0 for b in taken)
    ops.reset_accumulators()
    assert not ops._accum_reserve


def test_larger_requests_than_a_share_are_cleared_in_the_graph(gpu, monkeypatch):
    from uniql_amd import ops
    call = _call(16, 1024, 8192, 13, gpu)
    ops.reset_accumulators()
    want = call().clone()
    monkeypatch.setattr(ops, "_RESERVE_SHARE", 1024)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = call()
    for _ in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    assert ops._accum_reserve[gpu.index][1] == 0
    ops.reset_accumulators()


@pytest.mark.parametrize("m", [1, 8, 12, 16])
def test_a_call_that_exchanges_nothing_takes_no_words(gpu, monkeypatch, m):
    """a workgroup per strip over all of K: neither words of the reserve nor a clearing kernel in the graph"""
    from uniql_amd import ops
    lib = ops._capi.load()
    monkeypatch.setattr(lib, "uniql_clear", lambda *a: pytest.fail("a clear in the graph"))
    call = _call(m, 4096, 28672, 14, gpu)
    ops.reset_accumulators()
    want = call().clone()
    assert not ops._accum_cache
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = call()
    assert not ops._accum_in_capture
    for _ in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
