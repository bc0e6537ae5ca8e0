"""Rows and graphs at the lines where the integer variants and SpMV codes
change between the direct, the binned and their own kernels: whole numbers, so
every route is equal to the oracle to the bit."""
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
def test_long_integer_rows_of_the_direct_pull(degrees):
    _check(*_rows(degrees, 30_011, sum(degrees)))
