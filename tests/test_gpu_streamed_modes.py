"""The direct and binned pulls in the other variants' arithmetic: integer sums
bit-exact against the oracle, the fp32 push within the reference's own spread
(1e-5) -- and, since its destinations add in source order here, equal to the
sequential pull.  Sizes: the direct pull's and, past 8 M edges, the binned
one's ("large", and "binned edges" with rows at its bins' and pieces' ends);
rows at the edges of a thread's, a wavefront's and a block's in the direct
one."""
import numpy as np
import pytest

import opengraph_amd as og
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

CAP = 19968      # in-edge values of a block's LDS
WAVES = [127, 128, 129, 511, 512, 513]   # the direct pull's thread rows: up to 128 integers, 512 fp32


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
        return _rows(1, [CAP - 1, CAP, CAP + 1, 2 * CAP + 5] + WAVES + [7] * 600 + [1] * 900, 20_003)
    if kind == "small":
        return og.rmat_host(12, 50_000, seed=4)
    if kind == "binned edges":    # bins of 4.6 k in-edges
        deg = [CAP - 1, CAP, CAP + 1, 2 * CAP, 2 * CAP + 1, 4600, 2300, 2301, 513] + WAVES
        return _rows(2, deg + [9] * 900_000 + [1] * 900_000, 2_000_003)
    return og.rmat_host(19, 9_000_000, seed=7)


@pytest.mark.parametrize("kind", ["edges", "small", "large", "binned edges"])
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


@pytest.mark.parametrize("kind", ["edges", "small", "large", "binned edges"])
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
