"""Edges of the build kernels (radix sort tiles, row copies, binned layout)
against numpy and the oracle: whole numbers, so everything is equal to the
bit.  The layout itself is checked index by index on the host before its
first launch (OG_BIN_VERIFY, set by conftest.py)."""
import numpy as np
import pytest

import opengraph_amd as og
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

TILE = 4096          # items of a radix sort tile
MAX_BLOCKS = 2048    # sort blocks; more tiles than that share blocks


@pytest.fixture(scope="module", autouse=True)
def device():
    og.init(0)


@pytest.mark.parametrize("edges", [1, 63, 64, 65, 1023, 1024, 1025, TILE - 1, TILE, TILE + 1, 3 * TILE + 1,
                                   MAX_BLOCKS * TILE + 5])
@pytest.mark.parametrize("ids", ["uniform", "one", "few"])
def test_stable_sort_at_tile_edges(edges, ids):
    """Forward list by source (stable), inverse list by destination of that."""
    rng = np.random.default_rng(edges)
    n = {"uniform": 70_001, "one": 1, "few": 3}[ids]
    s = rng.integers(0, n, edges).astype(np.uint32)
    d = rng.integers(0, 70_001, edges).astype(np.uint32)
    d[0] = 70_000
    g = og.Graph.from_edges(s, d, 0)
    o = np.argsort(s, kind="stable")
    fs, fd = s[o], d[o]
    i = np.argsort(fd, kind="stable")
    assert np.array_equal(g.array("f_src"), fs) and np.array_equal(g.array("f_dst"), fd)
    assert np.array_equal(g.array("i_src"), fd[i]) and np.array_equal(g.array("i_dst"), fs[i])
    g.free()


@pytest.mark.parametrize("edges", [1, 2, 3, 4, 5, 7, 8, 9, 4099, 300_002])
@pytest.mark.parametrize("ids", [1, 3, 50_000])
def test_mapping_at_quad_edges(edges, ids):
    """Run starts and lengths of the sorted keys: runs within, across and
    exactly of the four keys a thread reads, and no key at all."""
    rng = np.random.default_rng(edges + ids)
    s, d = (rng.integers(0, ids, edges).astype(np.uint32) for _ in range(2))
    s[-1] = ids - 1
    g = og.Graph.from_edges(s, d, 0)
    n = g.num_vertices
    for side, key in (("f", s), ("i", d)):
        deg = np.bincount(key, minlength=n)
        start = np.where(deg > 0, np.concatenate([[0], np.cumsum(deg)[:-1]]), 0)
        assert np.array_equal(g.array(side + "_out_degree"), deg)
        assert np.array_equal(g.array(side + "_edges_idx"), start)
    g.free()


@pytest.mark.parametrize("relabel", [0, 1, 2])
@pytest.mark.parametrize("degrees", [[1], [16, 17], [511, 512, 513], [4095, 4096, 4097], [19968], [19969, 1],
                                     [19967, 1, 1, 40000]])
def test_layout_at_row_class_edges(relabel, degrees):
    """Rows of exactly these in-degrees (the plan's and the layout's class
    boundaries), ordered by in-degree or left in their own order."""
    rng = np.random.default_rng(len(degrees) + degrees[0])
    n = 45_000
    dst = np.repeat(rng.permutation(n)[:len(degrees)], degrees)
    src = rng.integers(0, n, len(dst))
    src[0] = n - 1
    src, dst = src.astype(np.uint32), dst.astype(np.uint32)
    g = og.Graph.from_edges(src, dst, 0)
    ref = po.pagerank(po.build_csr(src, dst, 0, 4), 0, 0.0, 6, 4)
    pr = og.PageRank(g, 0, 6, 0.0, relabel=relabel, binned=1)
    pr.run()
    assert np.array_equal(pr.ranks().view(np.uint32), ref["ranks"].view(np.uint32))
    pr.free()
    g.free()


def test_layout_over_more_segments_than_one_window():
    """More than 4096 segments of 39,936 sources: the layout's kernels take
    them in windows.  Two iterations, against the pull that gathers (every
    row in CSR order)."""
    n = 4098 * 39_936 + 7
    rng = np.random.default_rng(11)
    e = 200_000
    src = rng.integers(0, n, e).astype(np.uint32)
    dst = rng.choice(rng.integers(0, n, 5000), e).astype(np.uint32)
    src[:4] = (0, n - 1, 4096 * 39_936, 4096 * 39_936 - 1)
    g = og.Graph.from_edges(src, dst, 0)
    out = []
    for kw in (dict(binned=1), dict(binned=2, hub_threshold=0xFFFFFFFF)):
        pr = og.PageRank(g, 0, 2, 0.0, **kw)
        pr.run()
        out.append(pr.ranks()[np.unique(dst)])
        pr.free()
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    g.free()
