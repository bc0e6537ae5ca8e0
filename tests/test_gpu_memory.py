"""Device memory that is handed out again, and results taken to the host by
several threads: what comes back is what was put in, to the bit."""
import threading

import numpy as np
import pytest

import opengraph_amd as og
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

PIECE = 1 << 18      # 32-bit words of a download's piece; 4 pieces and more go by threads
THREADS = 8


@pytest.fixture(scope="module", autouse=True)
def device():
    og.init(0)


def _csr(n, edges, rng):
    s, d = (rng.integers(0, n, edges).astype(np.uint32) for _ in range(2))
    return po.build_csr(s, d, 0, 4), s, d


@pytest.mark.parametrize("words", [1, 4 * PIECE - 1, 4 * PIECE, 4 * PIECE + 1, THREADS * PIECE - 1,
                                   THREADS * PIECE + 1, 17 * PIECE + 3])
def test_download_at_piece_edges(words):
    rng = np.random.default_rng(words)
    s, d = (np.sort(rng.integers(0, 1 << 20, words)).astype(np.uint32) for _ in range(2))
    g = og.Graph.from_edges(s, d, 0)
    for _ in range(2):
        assert np.array_equal(g.array("f_src"), s) and np.array_equal(g.array("f_dst"), d)
    g.free()


def test_reused_blocks_hold_nothing():
    """Graphs and states of changing sizes in the blocks of the ones before."""
    rng = np.random.default_rng(0)
    for n, e in [(5000, 60_000), (4900, 59_000), (70_000, 300_000), (5000, 60_000), (100, 90_000), (70_001, 299_999)]:
        c, s, d = _csr(n, e, rng)
        ref = po.pagerank(c, 0, 0.0, 5, 4)
        g = og.Graph.from_edges(s, d, 0)
        pr = og.PageRank(g, 0, 5, 0.0)
        for _ in range(2):
            pr.run()
            assert np.array_equal(pr.ranks().view(np.uint32), ref["ranks"].view(np.uint32))
        pr.free()
        g.free()


def test_threads_share_the_blocks():
    rng = np.random.default_rng(1)
    work = []
    for n, e in [(3000, 40_000), (3100, 40_500), (60_000, 200_000), (1_500_000, 1_600_000)]:
        c, s, d = _csr(n, e, rng)
        work.append((s, d, po.pagerank(c, 0, 0.0, 4, 4)["ranks"].view(np.uint32)))
    bad = []

    def run(s, d, want):
        try:
            for _ in range(4):
                g = og.Graph.from_edges(s, d, 0)
                pr = og.PageRank(g, 0, 4, 0.0)
                pr.run()
                if not np.array_equal(pr.ranks().view(np.uint32), want):
                    bad.append(len(s))
                pr.free()
                g.free()
        except Exception as e:          # a thread's failure is the test's
            bad.append(e)

    th = [threading.Thread(target=run, args=w) for w in work]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
