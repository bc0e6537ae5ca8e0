"""The work that users of opengraph_amd have it do, as cases to be timed.

Every case is one call sequence of the public Python API on a graph made from
a seed.  R-MAT graphs (a, b, c = 0.57, 0.19, 0.19, ids permuted) stand for
the power-law graphs that PageRank is run on, uniform graphs for meshes of
random links; the sizes run from a graph that fits one compute unit's LDS to
the 2^24-vertex, 2^28-edge benchmark graph.

Kinds:
  pagerank  a graph kept on the device, ranked again and again (a driver that
            sweeps variants and options): PageRank.run, then the ranks.
  edges     an edge list on the device to ranks: Graph.build, the run's plan,
            the iterations, the ranks (a graph that is ranked once).
  ppr       a kept graph queried with k restart vertices: Ppr, run, ranks.
  multi     a kept batch of uneven graphs ranked in one hipGraph launch.
  spmv      the SpMV benchmark on a kept graph.
  learned   a kept graph and a kept trained network: the learned start, the
            iterations to an L1 change below epsilon, the ranks.
"""
import ctypes
import math
import warnings

import numpy as np
import torch

import opengraph_amd as og

DAMP = 0.85
BASE = float(np.float32(1.0) - np.float32(DAMP))


# ----------------------------------------------------------------- the cases

def _pagerank(graph, vertices, edges, variant, iterations, epsilon):
    return dict(kind="pagerank", graph=graph, vertices=vertices, edges=edges, variant=variant,
                iterations=iterations, epsilon=epsilon)


def _edges(graph, vertices, edges, sort, iterations):
    return dict(kind="edges", graph=graph, vertices=vertices, edges=edges, sort=sort, iterations=iterations)


def _ppr(vertices, edges, k, iterations):
    return dict(kind="ppr", graph="rmat", vertices=vertices, edges=edges, k=k, iterations=iterations)


def _multi(graphs, low, high, iterations):
    return dict(kind="multi", graphs=graphs, low=low, high=high, iterations=iterations)


def _spmv(graph, vertices, edges, code, iterations):
    return dict(kind="spmv", graph=graph, vertices=vertices, edges=edges, code=code, iterations=iterations)


def _learned(vertices, edges, epsilon):
    return dict(kind="learned", graph="rmat", vertices=vertices, edges=edges, epsilon=epsilon)


def listed():
    return [
        # a small graph ranked at the reference's defaults (-p 0, 20 iterations): launches and latency
        dict(_pagerank("rmat", 1 << 10, 12345, 0, 20, 1e-4), name="pull_1k"),
        # the R-MAT scale 16 graph of the tests, iterated until no vertex moves by 1e-6
        dict(_pagerank("rmat", 1 << 16, 1 << 20, 0, 100, 1e-6), name="pull_rmat16_converge"),
        # a uniform graph with an odd vertex count, every source as often gathered as any other
        dict(_pagerank("uniform", 3000017, 40000003, 0, 20, 1e-4), name="pull_uniform_3m"),
        # the benchmark's graph: R-MAT scale 24, edge factor 16
        dict(_pagerank("rmat", 1 << 24, 1 << 28, 0, 20, 1e-4), name="pull_rmat24"),
        # -p 1, the reference's push with fp32 atomics
        dict(_pagerank("rmat", 1 << 20, 1 << 24, 1, 20, 1e-4), name="push_rmat20"),
        # -p 2, the reference's fixed-point pull (u64 sums)
        dict(_pagerank("rmat", 1 << 22, 1 << 26, 2, 20, 1e-4), name="fixed_pull_rmat22"),
        # a small edge list sorted by destination too (-o 1), ranked once
        dict(_edges("rmat", 1 << 14, 200003, 1, 20), name="edges_small"),
        # a large edge list (-o 0) ranked once at the reference's defaults
        dict(_edges("rmat", 1 << 22, 1 << 26, 0, 20), name="edges_rmat22"),
        # a full batch of 64 personalized queries
        dict(_ppr(1 << 18, 1 << 22, 64, 20), name="ppr64_rmat18"),
        # the uneven batch, ten times smaller than the benchmark's 256 graphs
        dict(_multi(24, 12, 18, 50), name="multi_24"),
        # -a 5 -p 0: the SpMV benchmark's 20 passes
        dict(_spmv("rmat", 1 << 21, 1 << 25, 0, 20), name="spmv_rmat21"),
        # a trained start on a graph larger than those it was trained on
        dict(_learned(1 << 21, 1 << 25, 1e-6), name="learned_rmat21"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pagerank", "pagerank", "pagerank", "edges", "edges", "ppr", "multi", "spmv", "learned"])
    graph = rng.choice(["rmat", "rmat", "uniform"])
    if kind == "multi":
        low = rng.randint(10, 13)
        return _multi(rng.randint(2, 32), low, rng.randint(low + 1, 18), rng.randint(10, 60))
    top = {"pagerank": 1 << 26, "edges": 1 << 26, "ppr": 1 << 23, "spmv": 1 << 26, "learned": 1 << 25}[kind]
    edges = log(5000, top)
    vertices = max(300, int(edges / math.exp(rng.uniform(math.log(4), math.log(40)))))
    if kind == "ppr":
        return _ppr(vertices, edges, rng.choice([1, 2, 5, 17, 32, 33, 50, 64]), rng.randint(8, 30))
    if kind == "learned":
        return _learned(vertices, edges, 1e-6)
    if kind == "edges":
        return _edges(graph, vertices, edges, rng.choice([0, 1]), rng.randint(5, 40))
    if kind == "spmv":
        return _spmv(graph, vertices, edges, rng.choice([0, 0, 1, 2, 3]), rng.randint(5, 30))
    return _pagerank(graph, vertices, edges, rng.choice([0, 0, 0, 1, 2, 3, 4]), rng.randint(5, 60), 1e-4)


# ---------------------------------------------------------------- the inputs

class _Borrowed:
    """A device array that torch owns, as the edge arrays of Graph.build."""

    def __init__(self, t):
        self.tensor = t
        self.nbytes = t.numel() * t.element_size()
        self.ptr = ctypes.c_void_p(t.data_ptr())


def _edge_list(graph, vertices, edges, seed):
    """Two int32 tensors of vertex ids in [0, vertices); the largest id is
    always vertices - 1, so that the vertex count is the one asked for."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if graph == "uniform":
        src = torch.randint(0, vertices, (edges,), device="cuda", dtype=torch.int32, generator=gen)
        dst = torch.randint(0, vertices, (edges,), device="cuda", dtype=torch.int32, generator=gen)
    else:
        src = torch.zeros(edges, device="cuda", dtype=torch.int32)
        dst = torch.zeros(edges, device="cuda", dtype=torch.int32)
        u = torch.empty(edges, device="cuda", dtype=torch.float32)
        for _ in range(max(1, (vertices - 1).bit_length())):
            u.uniform_(0, 1, generator=gen)
            low = u >= 0.57 + 0.19
            src.mul_(2).add_(low)
            dst.mul_(2).add_(((u >= 0.57) & ~low) | (u >= 0.57 + 0.19 + 0.19))
        del u
        perm = torch.randperm(vertices, device="cuda", generator=gen, dtype=torch.int32)
        for a in (src, dst):
            # (ids past a vertex count that is no power of two fold back)
            a.remainder_(vertices)
            a.copy_(perm[a])
    src[0] = vertices - 1
    return src, dst


def _prepared_graph(case, seed, sort=0):
    src, dst = _edge_list(case["graph"], case["vertices"], case["edges"], seed)
    torch.cuda.synchronize()
    return og.Graph.build(_Borrowed(src), _Borrowed(dst), case["edges"], sort)


def _sources(case, seed):
    """k distinct restart vertices that have out-edges."""
    src, _ = _edge_list(case["graph"], case["vertices"], case["edges"], seed)
    ids = torch.unique(src).cpu().numpy()
    rng = np.random.default_rng(seed)
    return rng.choice(ids, size=case["k"], replace=len(ids) < case["k"]).astype(np.uint32)


def _batch(case, seed):
    """(vertices, edges, seed) of each graph of a batch: sizes spread evenly over the scales, edge
    factors over 8 to 32."""
    rng = np.random.default_rng(1000 + case["graphs"])  # the sizes belong to the case, the edges to the seed
    n = case["graphs"]
    scales = np.linspace(case["low"], case["high"], n)
    got = []
    for i in range(n):
        v = int(2 ** scales[i])
        got.append((v, int(v * rng.uniform(8, 32)), seed * 1000 + i))
    return got


_TRAIN_SEED = 99


def _trained():
    """The network a program has trained once: on one small graph, a few epochs."""
    m = og.Mlp(seed=1)
    src, dst = _edge_list("rmat", 1 << 14, 1 << 18, _TRAIN_SEED)
    torch.cuda.synchronize()
    g = og.Graph.build(_Borrowed(src), _Borrowed(dst), 1 << 18, 0)
    m.add_graph(g, tol=1e-9, max_iter=200)
    m.train(epochs=4, batch=4096, lr=3e-3, seed=1)
    g.free()
    return m


def prepare(case, seed):
    og.init(0)
    kind = case["kind"]
    s = {"case": case}
    if kind == "edges":
        s["src"], s["dst"] = (_Borrowed(t) for t in _edge_list(case["graph"], case["vertices"], case["edges"], seed))
        torch.cuda.synchronize()
    elif kind == "multi":
        s["graphs"] = [_prepared_graph(dict(graph="rmat", vertices=v, edges=e), sd) for v, e, sd in _batch(case, seed)]
        # a fixed row split and tile shape: a batch whose results must not depend on a timing
        s["run"] = og.Multi(s["graphs"], max_iter=case["iterations"], epsilon=1e-6, hub_threshold=16,
                            hub_thresholds=[16] * case["graphs"], tiles=[(256, 4, 8)] * case["graphs"])
    else:
        s["graph"] = _prepared_graph(case, seed)
        if kind == "pagerank":
            s["run"] = og.PageRank(s["graph"], variant=case["variant"], max_iter=case["iterations"],
                                   epsilon=case["epsilon"])
        elif kind == "ppr":
            s["sources"] = _sources(case, seed)
        elif kind == "spmv":
            s["run"] = og.Spmv(s["graph"], code=case["code"])
        elif kind == "learned":
            s["mlp"] = _trained()
            s["run"] = og.PageRank(s["graph"], max_iter=200, epsilon=case["epsilon"], stop_rule=1, init_mode=1)
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "pagerank":
        s["run"].run()
        return s["run"].ranks()
    if kind == "edges":
        g = og.Graph.build(s["src"], s["dst"], case["edges"], case["sort"])
        pr = og.PageRank(g, max_iter=case["iterations"])
        pr.run()
        out = pr.ranks()
        pr.free()
        g.free()
        return out
    if kind == "ppr":
        p = og.Ppr(s["graph"], s["sources"], max_iter=case["iterations"], epsilon=1e-9)
        p.run()
        out = p.ranks()
        p.free()
        return out
    if kind == "multi":
        s["run"].run(mode=2)
        return [s["run"].result(i)[1] for i in range(case["graphs"])]
    if kind == "spmv":
        s["run"].run(case["iterations"])
        return s["run"].output()
    s["run"].set_init_learned(s["mlp"])
    s["run"].run()
    return s["run"].ranks()


# ------------------------------------------- what a pass cannot do without

def work(case):
    """Per iteration each in-edge's source index and each vertex's row
    offset, contribution read and contribution written; the edge list twice
    over (read, and both CSRs written) where the pass builds the graph; the
    outputs once.  One multiply-add an edge and column."""
    kind = case["kind"]
    if kind == "multi":
        e = sum(x[1] for x in _batch(case, 1))
        n = sum(x[0] for x in _batch(case, 1))
    else:
        e, n = case["edges"], case["vertices"]
    k = case.get("k", 1)
    it = case.get("iterations") or 12  # the learned start's iterations
    per = {"pagerank": 4 * e + 12 * n, "edges": 4 * e + 12 * n, "multi": 4 * e + 12 * n, "learned": 4 * e + 12 * n,
           "spmv": 4 * e + 12 * n, "ppr": 4 * e + 4 * n + 8 * n * k}[kind]
    if case.get("variant") in (2, 3) or case.get("code") in (2, 3):
        per += 8 * n  # 64-bit contributions
    extra = 4 * n * k
    if kind == "edges":
        extra += 8 * e + 16 * e + 24 * n
    if kind == "learned":
        extra += 4 * e + 24 * n
    flops = 2.0 * e * k * it + (8832.0 * n if kind == "learned" else 0)
    return {"bytes": float(per) * it + extra, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("pagerank", "edges") and case.get("variant", 0) != 1:
        # the fp32 pull adds every row in the reference's order, the others add whole numbers
        return "exact"
    if kind == "spmv" and case["code"] != 1:
        return "exact"
    if kind in ("ppr", "multi"):
        # rows of hundreds of in-edges in fp32 trees: 1.2e-7 to 2.3e-7 from the 64-bit result
        return {"rel": 1e-6, "max": 2e-5}
    # running fp32 sums over up to 10^5 in-edges: the push and the SpMV push in any order (7.6e-6 from
    # the 64-bit result, 1.4e-7 between two runs), the learned start's iterations (1.2e-5 from the fixed
    # point at their stop)
    return {"rel": 3e-5, "max": 3e-4}


# ------------------------------------------------------------ 64-bit results

def _pull_matrix(src, dst, n, weight):
    """The n x n matrix with weight[u] at (v, u) for every edge (u, v), in 64 bits."""
    order = torch.argsort(dst)
    cols = src[order].contiguous()
    del order
    rows = torch.zeros(n + 1, device="cuda", dtype=torch.int32)
    rows[1:] = torch.bincount(dst, minlength=n).cumsum(0)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")  # torch calls its sparse tensors beta
        return torch.sparse_csr_tensor(rows, cols, weight[cols], (n, n), check_invariants=False)


def _out_degree(src, n):
    return torch.bincount(src, minlength=n).double()


def _pagerank64(src, dst, n, iterations, epsilon, l1=False, start=BASE):
    a = _pull_matrix(src, dst, n, DAMP / _out_degree(src, n).clamp(min=1))
    x = torch.full((n, 1), start, device="cuda", dtype=torch.float64)
    for _ in range(iterations):
        new = BASE + a @ x
        change = (new - x).abs()
        x = new
        if (float(change.sum()) / n < epsilon) if l1 else not bool((change >= epsilon).any()):
            break
    return x[:, 0] / n


def exact(case, seed):
    kind = case["kind"]
    if kind == "multi":
        outs = []
        for v, e, sd in _batch(case, seed):
            src, dst = _edge_list("rmat", v, e, sd)
            outs.append(_pagerank64(src, dst, v, case["iterations"], 1e-6))
        return outs
    n = case["vertices"]
    src, dst = _edge_list(case["graph"], n, case["edges"], seed)
    if kind == "learned":
        # the fixed point that the iterations from any start end near
        return _pagerank64(src, dst, n, 200, 1e-10, l1=True, start=1.0)
    if kind == "ppr":
        at = torch.from_numpy(_sources(case, seed).astype(np.int64)).cuda()
        cols = torch.arange(case["k"], device="cuda")
        a = _pull_matrix(src, dst, n, DAMP / _out_degree(src, n).clamp(min=1))
        x = torch.zeros((n, case["k"]), device="cuda", dtype=torch.float64)
        x[at, cols] = 1.0
        restart = (1.0 - DAMP) * x
        live = torch.ones(case["k"], device="cuda", dtype=torch.bool)
        for _ in range(case["iterations"]):
            new = restart + a @ x
            change = (new - x).abs().sum(0)
            x = torch.where(live, new, x)
            live = live & (change >= 1e-9)
        return x
    if kind == "spmv":
        if case["code"] == 2:
            return None  # the Q16.16 terms (7 x) >> 16 are defined by their rounding down
        # (every gathered source has an out-edge, so no row sees the value of the others)
        a = _pull_matrix(src, dst, n, 1.0 / _out_degree(src, n).clamp(min=1))
        w = float(np.float32(0.0001))
        return case["iterations"] * w * (a @ torch.ones((n, 1), device="cuda", dtype=torch.float64))[:, 0]
    return _pagerank64(src, dst, n, case["iterations"], case.get("epsilon", 1e-4))
