"""The direct and binned pulls in the other variants' arithmetic: integer sums
bit-exact against the oracle, the fp32 push within the reference's own spread
(1e-5) -- and, since its destinations add in source order here, equal to the
sequential pull.  Sizes: the direct pull's and, past 8 M edges, the binned
one's; rows at the edges of a thread's, a wavefront's and a bin's."""
import numpy as np
import pytest

import opengraph_amd as og
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

CAP, WAVE = 19968, 192


@pytest.fixture(scope="module", autouse=True)
def device():
    og.init(0)


def _rows(seed, degrees, n):
    rng = np.random.default_rng(seed)
    dst = np.repeat(rng.permutation(n)[:len(degrees)], degrees).astype(np.uint32)
    src = rng.integers(0, n, len(dst)).astype(np.uint32)
    src[0] = n - 1
    return src, dst


def _graph(kind):
    if kind == "edges":
        return _rows(1, [CAP - 1, CAP, CAP + 1, 2 * CAP + 5, WAVE - 1, WAVE, WAVE + 1] + [7] * 600 + [1] * 900, 20_003)
    if kind == "small":
        return og.rmat_host(12, 50_000, seed=4)
    return og.rmat_host(19, 9_000_000, seed=7)


@pytest.mark.parametrize("kind", ["edges", "small", "large"])
def test_variants_against_the_oracle(kind):
    s, d = _graph(kind)
    g = og.Graph.from_edges(s, d, 0)
    o = po.build_csr(s, d, 0, 8)
    for code in (2, 3, 4, 9, 1):
        for eps, iters in ((0.0, 5), (1e-4, 60)):
            ref = po.pagerank(o, 0 if code == 1 else code, eps, iters, 8)
            pr = og.PageRank(g, code, iters, eps)
            res = pr.run()
            x = pr.ranks()
            act, err = pr.rows()
            assert np.array_equal(x.view(np.uint32), ref["ranks"].view(np.uint32)), (kind, code, eps)
            assert res.iterations == ref["iterations"] and list(act) == list(ref["active"]), (kind, code, eps)
            np.testing.assert_allclose(err, ref["errors"], rtol=1e-9, atol=0)
            pr.free()
    g.free()


@pytest.mark.parametrize("kind", ["edges", "small", "large"])
def test_spmv_codes_against_the_oracle(kind):
    s, d = _graph(kind)
    g = og.Graph.from_edges(s, d, 0)
    o = po.build_csr(s, d, 0, 8)
    for code in (0, 1, 2, 3):
        y0 = po.spmv(o, 0 if code == 1 else code, 3)
        sp = og.Spmv(g, code)
        for _ in range(2):
            sp.run(3)
            assert np.array_equal(sp.output().view(np.uint32), y0.view(np.uint32)), (kind, code)
        sp.free()
    g.free()
