"""Stream scratch and recorded graphs: a call recorded on a stream that has no
scratch yet gets memory that outlives its graph (not the graph's own), and a
kept buffer that a graph uses outlives its growth.

The scatter into several LDS windows leaves its spills in scratch (slot 0), the
grouped fp8 dot its tile prefix (slot 1).  Integer values: results are exact.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scatter(tx, dev, n, nbins, seed):
    """Buffers, a run and a check of a Zipf scatter-add (its keys spill)."""
    idx = torch.empty(n, dtype=torch.int32, device=dev)
    val = torch.empty(n, dtype=torch.int32, device=dev)
    bins = torch.empty(nbins, dtype=torch.int32, device=dev)
    g = np.random.default_rng(seed)
    cdf = np.cumsum(np.arange(1, nbins + 1, dtype=np.float64) ** -1.1)
    want = np.zeros(nbins, np.int64)

    def fresh():
        k = np.minimum(np.searchsorted(cdf, g.random(n) * cdf[-1], side="right"), nbins - 1).astype(np.int32)
        v = g.integers(-9, 10, n, dtype=np.int32)
        idx.copy_(torch.from_numpy(k)), val.copy_(torch.from_numpy(v)), bins.zero_()
        want[:] = np.bincount(k, weights=v, minlength=nbins).astype(np.int64)
        torch.cuda.synchronize()

    def check():
        torch.cuda.synchronize()
        assert np.array_equal(bins.cpu().numpy(), want)

    return (lambda: tx.atomic_rmw("add", bins, idx, val)), fresh, check


def _grouped(tx, dev, groups, seed):
    N, K, rows = 264, 256, 3
    g = torch.Generator().manual_seed(seed)
    M = groups * rows
    a = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=dev)
    b = torch.randint(-3, 4, (groups, N, K), generator=g).float()
    bq = b.to(torch.float8_e4m3fn).to(dev)
    off = (torch.arange(groups + 1, dtype=torch.int32) * rows).to(dev)
    sa, sb = torch.ones(M, device=dev), torch.ones(groups, N, device=dev)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    want = [None]

    def fresh():
        x = torch.randint(-3, 4, (M, K), generator=g).float()
        a.copy_(x.to(torch.float8_e4m3fn)), out.zero_()
        want[0] = torch.bmm(x.view(groups, rows, K), b.transpose(1, 2).contiguous()).view(M, N).to(torch.bfloat16)
        torch.cuda.synchronize()

    def check():
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), want[0])

    return (lambda: tx.dot_scaled_rowcol_grouped(a, sa, bq, sb, off, out=out)), fresh, check


def _cases(tx, dev):
    return [_scatter(tx, dev, 1 << 18, 65536, 1), _grouped(tx, dev, 20, 2), _scatter(tx, dev, 40_000, 100_000, 3),
            _grouped(tx, dev, 5, 4)]


def _eager(case):
    run, fresh, check = case
    fresh()
    run()
    check()


def _record(case, stream):
    graph = torch.cuda.CUDAGraph()
    case[1]()
    with torch.cuda.graph(graph, stream=stream):
        case[0]()
    return graph


def _replay(graph, case):
    case[1]()
    graph.replay()
    case[2]()


def test_recorded_without_scratch(tx, dev):
    """Recorded on a stream that never ran a call; graphs dropped one after
    another, the later ones and the eager calls after them are right."""
    cases = _cases(tx, dev)
    for c in cases:
        _eager(c)  # (on another stream: loads the kernels)
    side = torch.cuda.Stream()
    for c in cases:
        graph = _record(c, side)
        for _ in range(3):
            _replay(graph, c)
            _eager(cases[0])
        graph.reset()
        torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for c in cases + cases:
            _eager(c)


def test_recorded_scratch_outlives_growth(tx, dev):
    """Recorded with the stream's kept scratch, which eager calls then outgrow;
    the graph's replays and the eager calls stay right in turn."""
    small, large = _scatter(tx, dev, 40_000, 65536, 5), _scatter(tx, dev, 1 << 22, 65536, 6)
    _eager(large)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        _eager(small)
    before = tx.lib.txScratchAllocations()
    graph = _record(small, side)
    assert tx.lib.txScratchAllocations() == before  # the kept buffer, not one of the graph's
    _replay(graph, small)
    with torch.cuda.stream(side):
        _eager(large)
    assert tx.lib.txScratchAllocations() == before + 1
    for _ in range(3):
        _replay(graph, small)
        with torch.cuda.stream(side):
            _eager(large)
