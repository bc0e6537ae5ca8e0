"""The direct pull (og_dir.hip, the default for a small graph's -p 0) against
the oracle's sequential pull: every row is the reference's running fp32 sum,
so ranks, iteration counts and activeVertices are equal to the bit.  Sizes at
its edges: one block and many, groups of 32 blocks, rows at the boundaries
between a thread, a wavefront and the pieces of one block's LDS, batches of
in-edges, stops at the first, the last and no iteration."""
import numpy as np
import pytest

import opengraph_amd as og
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

CAP = 19968      # in-edge values of a block's LDS
EDGES = 4096     # in-edges a block aims at
BATCH = 12 * 512


@pytest.fixture(scope="module", autouse=True)
def device():
    og.init(0)


def _graph(n, degrees, seed):
    """Rows of the given in-degrees (the other vertices have none) from random sources."""
    rng = np.random.default_rng(seed)
    dst = np.repeat(rng.permutation(n)[:len(degrees)], degrees).astype(np.uint32)
    src = rng.integers(0, n, len(dst)).astype(np.uint32)
    src[0] = n - 1
    return src, dst


def _same(src, dst, eps, iters, **kw):
    g = og.Graph.from_edges(src, dst, 0)
    ref = po.pagerank(po.build_csr(src, dst, 0, 4), 0, eps, iters, 4)
    pr = og.PageRank(g, 0, iters, eps, **kw)
    for _ in range(2):   # (a run leaves nothing for the next)
        res = pr.run()
        assert np.array_equal(pr.ranks().view(np.uint32), ref["ranks"].view(np.uint32))
        assert res.iterations == ref["iterations"]
        act, err = pr.rows()
        assert list(act) == list(ref["active"])
        np.testing.assert_allclose(err, ref["errors"], rtol=1e-9, atol=0)
    pr.free()
    g.free()
    return res


@pytest.mark.parametrize("degrees", [
    [1], [1, 1, 1], [3] * 512, [3] * 513, [511, 512, 513, 514], [64, 65, 575, 1344, 2368, 2369],
    [EDGES - 1, EDGES, EDGES + 1], [BATCH - 1, BATCH, BATCH + 1, 2 * BATCH + 1], [CAP - 1, CAP, CAP + 1],
    [5 * CAP // 2, 7], [8] * 20_000, [40] * 3000 + [2] * 9000])
@pytest.mark.parametrize("relabel", [1, 0])   # by in-degree, and in the caller's order
def test_row_and_block_edges(degrees, relabel):
    src, dst = _graph(30_011, degrees, sum(degrees))
    _same(src, dst, 0.0, 7, relabel=relabel)


@pytest.mark.parametrize("edges", [32 * EDGES, 64 * EDGES - 5, 65 * EDGES, 300_000])
@pytest.mark.parametrize("eps,iters", [(1e-3, 200), (1e9, 5), (1e9, 1), (0.0, 1), (0.0, 2), (0.0, 257), (1e-12, 300)])
def test_stops_and_block_counts(edges, eps, iters):
    rng = np.random.default_rng(edges)
    n = edges // 7
    src = rng.integers(0, n, edges).astype(np.uint32)
    dst = rng.integers(0, n, edges).astype(np.uint32)
    src[0] = n - 1
    _same(src, dst, eps, iters)


def test_blocks_that_do_not_wait(monkeypatch):
    """With no polls allowed every block leaves at the first barrier; the run
    then goes one iteration a launch, to the same bits."""
    monkeypatch.setenv("OG_DIR_SPIN", "0")
    src, dst = og.rmat_host(14, 16 << 14, seed=5)
    _same(src, dst, 1e-5, 60)


@pytest.mark.parametrize("spin", [1, 33, 64, 200])
@pytest.mark.parametrize("iters", [60, 300])   # one launch, and launches of 256 iterations
def test_blocks_that_give_up(monkeypatch, spin, iters):
    """With a few polls some blocks give up at some barrier and the others leave
    with them; the same bits, and so in later runs, which try again."""
    monkeypatch.setenv("OG_DIR_SPIN", str(spin))
    src, dst = og.rmat_host(15, 16 << 15, seed=5)
    ref = po.pagerank(po.build_csr(src, dst, 0, 4), 0, 0.0, iters, 4)["ranks"].view(np.uint32)
    g = og.Graph.from_edges(src, dst, 0)
    pr = og.PageRank(g, 0, iters, 0.0)
    for _ in range(70):
        pr.run()
        assert np.array_equal(pr.ranks().view(np.uint32), ref)
    pr.free()
    g.free()


def test_enqueued_iterations_equal_a_run():
    src, dst = og.rmat_host(13, 16 << 13, seed=6)
    g = og.Graph.from_edges(src, dst, 0)
    pr = og.PageRank(g, 0, 9, 0.0)
    pr.run()
    want = pr.ranks()
    pr.reset()
    pr.enqueue(9, True)
    assert pr.kernel_ms()[1] == 9
    act, _ = pr.rows()
    pr.run()
    assert np.array_equal(pr.ranks(), want) and len(act) == 9
    pr.free()
    g.free()
