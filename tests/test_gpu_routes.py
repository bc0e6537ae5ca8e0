"""Rows and graphs at the lines where the integer variants and SpMV codes
change between the direct, the binned and their own kernels: whole numbers, so
every route is equal to the oracle to the bit."""
import time

import numpy as np
import pytest

import opengraph_amd as og
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

CAP = 19968      # in-edge values of a block's LDS
EDGES = 4096     # in-edges a block of the direct pull aims at
WAVE = 128       # rows of more in-edges are not added by one thread


@pytest.fixture(scope="module", autouse=True)
def device():
    og.init(0)


def _rows(degrees, n, seed):
    """Rows of the given in-degrees (the other vertices have none) from random sources."""
    rng = np.random.default_rng(seed)
    dst = np.repeat(rng.permutation(n)[:len(degrees)], degrees).astype(np.uint32)
    src = rng.integers(0, n, len(dst)).astype(np.uint32)
    src[0] = n - 1
    return src, dst


def _check(s, d, codes=(2, 3, 4, 9), spmv=(2, 3), relabel=1, iters=4):
    g = og.Graph.from_edges(s, d, 0)
    o = po.build_csr(s, d, 0, 8)
    for code in codes:
        ref = po.pagerank(o, code, 0.0, iters, 8)
        pr = og.PageRank(g, code, iters, 0.0, relabel=relabel)
        for _ in range(2):
            pr.run()
            assert np.array_equal(pr.ranks().view(np.uint32), ref["ranks"].view(np.uint32)), code
            assert list(pr.rows()[0]) == list(ref["active"]), code
        pr.free()
    for code in spmv:
        want = po.spmv(o, code, 3)
        sp = og.Spmv(g, code)
        sp.run(3)
        assert np.array_equal(sp.output().view(np.uint32), want.view(np.uint32)), code
        sp.free()
    g.free()


@pytest.mark.parametrize("degrees", [
    [WAVE - 1, WAVE, WAVE + 1], [WAVE + 1], [EDGES - 1, EDGES, EDGES + 1], [EDGES // 2] * 3, [511, 512, 513, 575],
    [CAP - 1, CAP, CAP + 1, CAP // 2], [CAP + 511, 1, 1], [2 * CAP, 2 * CAP + 1, 300] + [3] * 2000])
@pytest.mark.parametrize("relabel", [1, 0])
def test_long_integer_rows_of_the_direct_pull(degrees, relabel):
    _check(*_rows(degrees, 30_011, sum(degrees)), spmv=(2, 3) if relabel else (), relabel=relabel)


@pytest.mark.parametrize("relabel", [1, 0])
def test_integer_modes_past_the_direct_pull(relabel):
    s, d = og.rmat_host(18, 9_000_000, seed=3)
    _check(s, d, spmv=(), relabel=relabel, iters=3)


def _best(f, n=15):
    t = []
    for _ in range(n):
        a = time.perf_counter()
        f()
        t.append(time.perf_counter() - a)
    return min(t)


def _not_the_slower_form(s, d, codes, spmv, most=1.4, **opt):
    """A default run takes at most `most` times what the variant's own kernels
    take (binned = 2; SpMV: a hub_threshold); best of fifteen runs each, 20
    iterations."""
    g = og.Graph.from_edges(s, d, 0)
    for code in codes:
        t = []
        for kw in (dict(), dict(binned=2)):
            pr = og.PageRank(g, code, 20, 0.0, **opt, **kw)
            pr.run()
            t.append(_best(pr.run))
            pr.free()
        assert t[0] <= most * t[1], ("pagerank", code, t)
    for code in spmv:
        t = []
        for kw in (dict(), dict(hub_threshold=16)):
            sp = og.Spmv(g, code, **kw)
            sp.run(20)
            t.append(_best(lambda: sp.run(20)))
            sp.free()
        assert t[0] <= most * t[1], ("spmv", code, t)
    g.free()


def _hub(n, edges, hub, seed=3):
    """A uniform graph, `hub` of whose in-edges are one vertex's."""
    rng = np.random.default_rng(seed)
    s, d = (rng.integers(0, n, edges).astype(np.uint32) for _ in range(2))
    s[0] = n - 1
    d[:] = np.where(d == 7, 8, d)
    d[rng.permutation(edges)[:hub]] = 7
    return s, d


ROW = 24576      # an integer row that is always streamed; longer: a 40th of the in-edges


@pytest.mark.parametrize("edges,hub", [(300_000, ROW - 1), (300_000, ROW), (300_000, ROW + 1),
                                       (40 * ROW + 40, ROW + 1), (40 * ROW + 40, ROW + 2)])
def test_integer_rows_at_the_longest_streamed(edges, hub):
    s, d = _hub(20_000, edges, hub)
    assert np.bincount(d).max() == hub
    _check(s, d)
    g = og.Graph.from_edges(s, d, 0)
    pr = og.PageRank(g, 2, 2, 0.0)      # its bytes per iteration tell its passes
    streamed = hub <= max(ROW, edges // 40)
    n = g.num_vertices
    assert pr.bytes_per_iteration() == (8 * edges + 20 * n if streamed else 12 * edges + 24 * n)
    pr.free()
    g.free()


@pytest.mark.parametrize("n,edges,hub", [(1 << 20, 1 << 22, 1 << 21), (100_000, 1 << 20, 200_000),
                                         (1 << 18, 1 << 22, 1 << 18)])
def test_long_integer_rows_are_not_one_blocks_work(n, edges, hub):
    _not_the_slower_form(*_hub(n, edges, hub), codes=(2, 4, 9), spmv=(2, 3))


@pytest.mark.parametrize("n,edges", [(4098, 4098 * 2048 + 2047), (4097, 4098 * 2048)])
def test_integer_pulls_of_few_vertices(n, edges):
    """Past 8 M edges (no direct pull) at and past 2048 in-edges a vertex."""
    rng = np.random.default_rng(n)
    s, d = (rng.integers(0, n, edges).astype(np.uint32) for _ in range(2))
    s[0] = n - 1
    _check(s, d, iters=3)
    g = og.Graph.from_edges(s, d, 0)
    pr = og.PageRank(g, 2, 2, 0.0)
    assert pr.bytes_per_iteration() == (8 * edges + 20 * n if edges // 2048 <= n else 12 * edges + 24 * n)
    pr.free()
    g.free()
    if n == 4097:
        _not_the_slower_form(s, d, codes=(2, 4, 9), spmv=(2, 3), most=1.2)


@pytest.mark.parametrize("edges", [(1 << 21) - 1, 1 << 21])
def test_quantized_pull_at_its_first_streamed_size(edges):
    _check(*og.rmat_host(17, edges, seed=8), codes=(4,), spmv=())


@pytest.mark.parametrize("scale", [4, 12, 14, 16])
def test_small_quantized_pull_is_not_the_slower_form(scale):
    _not_the_slower_form(*og.rmat_host(scale, 16 << scale, seed=9), codes=(4,), spmv=(), most=1.2)


def _permutation(n, seed=5):
    s = np.arange(n, dtype=np.uint32)
    return s, np.random.default_rng(seed).permutation(n).astype(np.uint32)


def test_short_rows_over_many_segments():
    """One in-edge a vertex from all over 2^24 others: 9 padded entries an edge."""
    s, d = _permutation(1 << 24)
    g = og.Graph.from_edges(s, d, 0)
    pr = og.PageRank(g, 2, 2, 0.0)
    assert pr.bytes_per_iteration() == 12.0 * len(s) + 24.0 * len(s)   # its own kernels
    pr.free()
    sp = og.Spmv(g, 1)
    assert sp.bytes_per_iteration() == 10.0 * len(s) + 8.0 * len(s)
    sp.free()
    g.free()
    _not_the_slower_form(s, d, codes=(1, 2, 3, 4, 9), spmv=(1, 2, 3), most=1.2)


@pytest.mark.parametrize("n", [6_000_000, 9_000_000])   # below and above 5.5 entries an edge
def test_short_rows_streamed_or_not(n):
    s, d = _permutation(n)
    _check(s, d, iters=2)
    g = og.Graph.from_edges(s, d, 0)
    pr = og.PageRank(g, 2, 2, 0.0)
    assert pr.bytes_per_iteration() == ((8.0 + 20.0) * n if n == 6_000_000 else (12.0 + 24.0) * n)
    pr.free()
    # every sum has one term: the push is the oracle's pull to the bit
    ref = po.pagerank(po.build_csr(s, d, 0, 8), 0, 0.0, 3, 8)["ranks"]
    pr = og.PageRank(g, 1, 3, 0.0)
    pr.run()
    assert np.array_equal(pr.ranks().view(np.uint32), ref.view(np.uint32))
    pr.free()
    g.free()


@pytest.mark.parametrize("kind", ["ring", "tree"])
def test_spmv_push_over_rows_of_one_in_edge(kind):
    n = 1 << 20
    v = np.arange(1, n, dtype=np.uint32)
    u = v - 1 if kind == "ring" else (np.random.default_rng(2).random(n - 1) * v).astype(np.uint32)
    s, d = u.astype(np.uint32), v
    g = og.Graph.from_edges(s, d, 0)
    sp = og.Spmv(g, 1)
    assert sp.bytes_per_iteration() == 10.0 * len(s) + 8.0 * n    # the partitioned scatter
    sp.run(3)
    want = po.spmv(po.build_csr(s, d, 0, 8), 0, 3)
    assert np.array_equal(sp.output().view(np.uint32), want.view(np.uint32))   # one term a row
    sp.free()
    g.free()
    _not_the_slower_form(s, d, codes=(), spmv=(1,), most=1.15)


@pytest.mark.parametrize("relabel", [0, 1])
@pytest.mark.parametrize("n,row", [(30_011, 4096 // 6), (8_000_000, 2048)])   # bins of 4096, and of more than 12288
def test_wavefront_rows_of_the_binned_pull(n, row, relabel):
    """Rows at the most in-edges that one thread adds, and at the steps of a wavefront's sum."""
    deg = [row - 1, row, row + 1, row + 2, 64 + 64 * 36, 64 + 64 * 36 + 1, 64 + 64 * 12, 64 + 64 * 12 + 1, 3] + [1] * 700
    s, d = _rows(deg, n, row)
    o = po.build_csr(s, d, 0, 8)
    ref = po.pagerank(o, 0, 0.0, 4, 8)["ranks"]
    g = og.Graph.from_edges(s, d, 0)
    pr = og.PageRank(g, 0, 4, 0.0, relabel=relabel, binned=1)
    pr.run()
    assert np.array_equal(pr.ranks().view(np.uint32), ref.view(np.uint32))
    pr.free()
    g.free()


def test_long_rows_in_small_bins_are_not_a_threads():
    """10 k rows of 900 terms, in bins of 4608: the SpMV's pass takes about what
    its bytes take (half as long again when threads added them)."""
    rng = np.random.default_rng(4)
    n, e = 10_000, 9 << 20
    s, d = (rng.integers(0, n, e).astype(np.uint32) for _ in range(2))
    g = og.Graph.from_edges(s, d, 0)
    t = []
    for code in (0, 2):      # fp32 in order, and u64 sums over the same layout
        sp = og.Spmv(g, code)
        sp.run(20)
        t.append(_best(lambda: sp.run(20)))
        sp.free()
    assert t[0] <= 1.3 * t[1], t
    g.free()


@pytest.mark.parametrize("kind", ["rmat", "hub", "tree"])
def test_dropin_calls_share_their_plans(kind, monkeypatch, capfd):
    """The drop-in entry points on one graph: each of the two plans is built by
    the first call that needs it and by no later one."""
    monkeypatch.setenv("OGPU_TRACE", "1")
    if kind == "rmat":
        s, d = og.rmat_host(13, 16 << 13, seed=7)
    elif kind == "hub":      # -p 2 and 3 by their own kernels
        s, d = _hub(20_000, 300_000, ROW + 1)
    else:                    # -p 1 scatters
        d = np.arange(1, 400_000, dtype=np.uint32)
        s = (np.random.default_rng(2).random(len(d)) * d).astype(np.uint32)
    o = po.build_csr(s, d, 0, 8)
    host = og.HostGraphCSR(o.a)

    def built():
        return capfd.readouterr().err.count("plan built")

    own = {"rmat": (), "hub": (2, 3), "tree": (1,)}[kind]
    built()
    plans = 0
    for code in (0, 1, 2, 3, 0, 1, 2, 3):
        y = og.spmv_graph_csr(host, code, 3)[0]
        if code == 1:
            np.testing.assert_allclose(y, po.spmv(o, 0, 3), rtol=1e-4)
        else:
            assert np.array_equal(y.view(np.uint32), po.spmv(o, code, 3).view(np.uint32)), code
        plans += built()
    assert plans == 1 + (1 if own else 0)
    ranks = og.pagerank_graph_csr(host, 0, 5, 0.0)[0]
    assert np.array_equal(ranks.view(np.uint32), po.pagerank(o, 0, 0.0, 5, 8)["ranks"].view(np.uint32))
    assert built() == 0
    for first in (True, False):
        for code in (1, 2, 3, 9):
            ranks = og.pagerank_graph_csr(host, code, 5, 0.0)[0]
            want = po.pagerank(o, 0 if code == 1 else code, 0.0, 5, 8)["ranks"]
            np.testing.assert_allclose(ranks, want, rtol=1e-5 if code == 1 else 0, atol=0)
        n = built()
        assert n == 0 or (first and n == 1)


@pytest.mark.parametrize("n", [1 << 14, (1 << 14) + 1])
@pytest.mark.parametrize("edges", [3 << 20, (3 << 20) + 1, 6 << 20, (6 << 20) + 1, 8 << 20, (8 << 20) + 1])
def test_largest_direct_graphs(n, edges):
    """Sizes around the direct pull's limits, SpMV's and the pulls', near and far."""
    rng = np.random.default_rng(edges)
    s, d = (rng.integers(0, n, edges).astype(np.uint32) for _ in range(2))
    s[0] = n - 1
    _check(s, d, codes=(2,) if edges <= (3 << 20) + 1 else (0, 9), spmv=(0, 2) if edges <= (3 << 20) + 1 else (), iters=2)


@pytest.mark.parametrize("scale", [14, 16])
def test_integer_pulls_in_the_callers_order(scale):
    _not_the_slower_form(*og.rmat_host(scale, 16 << scale, seed=9), codes=(2, 9), spmv=(), most=1.2, relabel=0)
