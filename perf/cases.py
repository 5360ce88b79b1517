"""Performance cases of the counting engine.

Each case is one call (or one served request mix) that a program makes
through the package's public entry points, on seeded synthetic graphs of the
families the package generates: RMAT (a/b/c/d = .57/.19/.19/.05),
Erdos-Renyi and Chung-Lu.  Graphs are resident before the call, as in a
program that counts several patterns on one graph; every output is an exact
integer.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the resident graphs and handles of a case
    run(state)          one call; returns the counts
    work(case)          bytes and operations the call cannot do without
    exact(case, seed)   None: outputs are whole numbers
"""

from __future__ import annotations

import math

import numpy as np

import openkhuzdulgraph_amd as kz
from openkhuzdulgraph_amd import _ffi, workloads

ABC = workloads.RMAT_ABC


def listed():
    return [
        # Triangles of an Erdos-Renyi graph given symmetric, as the apps load
        # it: short lists only, the call is launches and one light pass.
        dict(name="k3_er16", kind="clique", family="er", n=1 << 16, draws=1 << 20, sym=True, k=3),
        # The smallest call: a graph of a few thousand vertices, where the
        # latency of one launch sequence is what a caller sees.
        dict(name="k4_rmat12", kind="clique", family="rmat", scale=12, ef=16, sym=False, k=4),
        # The headline workload: 4-cliques of RMAT-24, edge factor 16.
        dict(name="k4_rmat24", kind="clique", family="rmat", scale=24, ef=16, sym=False, k=4),
        # 5-cliques, the deepest built-in pattern, at the ordinary size.
        dict(name="k5_rmat22", kind="clique", family="rmat", scale=22, ef=16, sym=False, k=5),
        # The level-by-level form of the clique plans.
        dict(name="plain_k4_rmat20", kind="plain", family="rmat", scale=20, ef=16, sym=False, k=4),
        # A plan of an application other than a clique: induced 3-vertex
        # motifs on the power-law graph of the census workload.
        dict(name="motif3_chunglu", kind="motif3", family="cl", n=4850000, draws=43000000, weight=20000, sym=True),
        # Induced 3- and 4-vertex census of the same graph.
        dict(name="census_chunglu", kind="census", family="cl", n=4850000, draws=43000000, weight=20000, sym=True),
        # Many uneven graphs, three patterns each, in one launch.
        dict(name="batch_pool64", kind="batch", graphs=64),
        # Labelled frequent subgraph mining, hundreds of candidate patterns.
        dict(name="fsm_chunglu", kind="fsm", family="cl", n=120000, draws=1000000, weight=2000, sym=True, labels=6,
             share=200),
        # Neighbour lists in host memory, an eighth of them at a time in HBM.
        dict(name="paged_k4_rmat18", kind="paged", family="rmat", scale=18, ef=16, sym=False, k=4, part=8),
        # Sorted-list intersections handed over as a batch of host arrays.
        dict(name="setops_8192", kind="setops", lists=2048, longest=2000, pairs=8192, op="intersect"),
        # A burst of queries on resident graphs, small ones among large ones.
        dict(name="serve_mix", kind="serve", pool=6, scale=20, queries=32),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _family(rng, lo, hi, families=("rmat", "er", "cl")):
    """A graph of about lo..hi draws (log-uniform) of a random family."""
    f = rng.choice(families)
    draws = _logint(rng, lo, hi)
    if f == "rmat":
        ef = rng.randint(8, 24)
        scale = max(10, min(22, int(round(math.log2(draws / ef)))))
        return dict(family="rmat", scale=scale, ef=max(1, min(24, draws >> scale)))
    deg = rng.uniform(16, 48)
    n = max(1000, int(2 * draws / deg)) | 1
    if f == "er":
        return dict(family="er", n=n, draws=draws)
    return dict(family="cl", n=n, draws=draws, weight=max(100, int(math.sqrt(n) * rng.uniform(2, 8))))


def _k(rng, graph, most):
    """A clique size; Erdos-Renyi graphs of these degrees hold triangles only."""
    return 3 if graph["family"] == "er" else rng.randint(3, most)


def draw(rng):
    kind = rng.choice(["clique", "clique", "clique", "plain", "motif3", "census", "batch", "fsm", "paged", "setops",
                       "serve"])
    if kind == "clique":
        c = _family(rng, 1 << 16, 1 << 26)
        return dict(kind=kind, **c, sym=rng.random() < 0.5, k=_k(rng, c, 5))
    if kind == "plain":
        c = _family(rng, 1 << 16, 1 << 24)
        return dict(kind=kind, **c, sym=rng.random() < 0.5, k=_k(rng, c, 4))
    if kind in ("motif3", "census"):
        return dict(kind=kind, **_family(rng, 1 << 16, 1 << 25, ("er", "cl")), sym=True)
    if kind == "batch":
        return dict(kind=kind, graphs=rng.randint(3, 64))
    if kind == "fsm":
        return dict(kind=kind, **_family(rng, 1 << 14, 1 << 20, ("er", "cl")), sym=True, labels=rng.randint(3, 8),
                    share=rng.randint(50, 400))
    if kind == "paged":
        c = _family(rng, 1 << 18, 1 << 22)
        return dict(kind=kind, **c, sym=False, k=_k(rng, c, 5), part=rng.randint(4, 16))
    if kind == "setops":
        return dict(kind=kind, lists=_logint(rng, 50, 2048), longest=_logint(rng, 20, 4000),
                    pairs=_logint(rng, 100, 8192) | 1, op=rng.choice(["intersect", "subtract", "intersect_count"]))
    return dict(kind="serve", pool=rng.randint(2, 6), scale=rng.randint(14, 20), queries=rng.randint(8, 32))


def _graph(case, seed, orient=None):
    """The case's graph, built in HBM (symmetric or degree-oriented)."""
    orient = (not case["sym"]) if orient is None else orient
    if case["family"] == "rmat":
        return kz.gpu_gen_rmat(case["scale"], case["ef"], *ABC, seed + 1, orient)
    if case["family"] == "er":
        return kz.gpu_gen_erdos_renyi(case["n"], case["draws"], seed + 1, orient)
    return kz.gpu_gen_chung_lu(case["n"], case["draws"], 2.3, case["weight"], seed + 1, orient)


def _motif3_plan():
    """Induced triangles (aggregator 0) and wedges (1) of a symmetric graph:
    every edge (v0, v1) in both directions; triangles from v0 < v1 by a third
    vertex above both, wedges centred at v0 by a leaf above v1."""
    p = _ffi.kz_plan_desc()
    p.pattern_size = 3
    p.num_aggregators = 2
    p.multiplicity[0] = p.multiplicity[1] = 1
    p.num_step_lists = 3
    for s in range(_ffi.KZ_MAX_PATTERN):
        for code in range(256):
            p.type_table[s][code] = 0xFF

    def ref(r, kind, a, b=0):
        r.kind, r.a, r.b = kind, a, b

    roots = p.lists[0]
    roots.num_ops, roots.num_outs = 0, 1
    o = roots.outs[0]
    o.kind, o.child_active, o.pred = _ffi.KZ_OUT_SCATTER, 1, 0b111
    ref(o.src, _ffi.KZ_SET_NBR, 0)
    p.type_table[1][0] = 0
    # order codes of (v0, v1): 2 is v0 < v1, 1 is v1 < v0
    up = p.lists[1]
    up.num_ops, up.num_outs = 2, 2
    down = p.lists[2]
    down.num_ops, down.num_outs = 1, 1
    for lst, ops in ((up, (_ffi.KZ_OP_INTERSECT, _ffi.KZ_OP_SUBTRACT)), (down, (_ffi.KZ_OP_SUBTRACT,))):
        for i, op in enumerate(ops):
            lst.ops[i].op = op
            ref(lst.ops[i].lhs, _ffi.KZ_SET_NBR, 0)
            ref(lst.ops[i].rhs, _ffi.KZ_SET_NBR, 1)
    for lst, slot, agg, pred in ((up, 0, 0, 1 << 4), (up, 1, 1, 1 << 4), (down, 0, 1, (1 << 2) | (1 << 4))):
        o = lst.outs[slot]
        o.kind, o.aggregator, o.pred = _ffi.KZ_OUT_COUNT, agg, pred
        ref(o.src, _ffi.KZ_SET_SLOT, 2, slot)
    p.type_table[2][2] = 1
    p.type_table[2][1] = 2
    return p


def _pool(seed, count, orient):
    """`count` graphs of the uneven pool, another stretch of it per seed."""
    first = (seed * 67) % workloads.POOL_SIZE
    return [workloads.pool_graph(kz, (first + 61 * i) % workloads.POOL_SIZE, gpu=True, orient=orient)
            for i in range(count)]


def _pairs(case, seed):
    """Sorted id lists of 1 .. `longest` ids (log-uniform lengths, the case's
    own; random gaps from the seed), the pairs of them and the id counts of
    the pairs' result slots."""
    shape = np.random.default_rng(case["pairs"])
    n = np.exp(shape.uniform(0, math.log(case["longest"]), case["lists"])).astype(np.int64)
    pairs = shape.integers(0, case["lists"], (case["pairs"], 2))
    rng = np.random.default_rng(seed)
    lists = [np.cumsum(rng.integers(1, 9, k)).astype(np.uint32) for k in n]
    slots = n[pairs[:, 0]] if case["op"] == "subtract" else np.minimum(n[pairs[:, 0]], n[pairs[:, 1]])
    return lists, [(int(a), int(b)) for a, b in pairs], int(slots.sum())


def prepare(case, seed):
    kz.init(0)
    kind = case["kind"]
    if kind in ("clique", "plain", "census"):
        return dict(kind=kind, g=_graph(case, seed), k=case.get("k"))
    if kind == "motif3":
        return dict(kind=kind, g=_graph(case, seed), plan=_motif3_plan())
    if kind == "batch":
        return dict(kind=kind, batch=kz.Batch(_pool(seed, case["graphs"], True), [3, 4, 5]))
    if kind == "fsm":
        g = _graph(case, seed)
        n = g.num_vertices
        g.set_labels(np.random.default_rng(seed).integers(0, case["labels"], n).astype(np.uint32))
        return dict(kind=kind, g=g, threshold=max(1, n // case["share"]))
    if kind == "paged":
        h = _graph(case, seed).download()
        nbytes = max(4 * h.num_entries // case["part"], 1 << 20)
        return dict(kind=kind, g=kz.PagedGraph(h, list_bytes=nbytes, cache_bytes=nbytes), k=case["k"])
    if kind == "setops":
        lists, pairs, ids = _pairs(case, seed)
        return dict(kind=kind, op=case["op"], lists=lists, pairs=pairs, ids=ids)
    # serve: triangles and 4-cliques of one larger graph, 5-cliques and
    # censuses of the pool, in a seeded order
    big = kz.gpu_gen_rmat(case["scale"], 16, *ABC, seed + 1, True)
    ori, sym = _pool(seed, case["pool"], True), _pool(seed, case["pool"], False)
    rng = np.random.default_rng(seed)
    queries = []
    for i in range(case["queries"]):
        j = int(rng.integers(0, case["pool"]))
        if i % 8 == 0:
            queries.append((big, "clique", 3 + (i // 8) % 2))
        else:
            queries.append((ori[j], "clique", 5) if rng.random() < 0.6 else (sym[j], "census", 0))
    return dict(kind=kind, server=kz.Server(hbm_budget=0, max_inflight=4), queries=queries)


def run(state):
    kind = state["kind"]
    if kind == "clique":
        return state["g"].count_cliques(state["k"], "persistent")
    if kind == "plain":
        return state["g"].count_cliques(state["k"], "plain")
    if kind == "motif3":
        return state["g"].count_plan(state["plan"])
    if kind == "census":
        return state["g"].motif_census()
    if kind == "batch":
        return state["batch"].run()
    if kind == "fsm":
        r = state["g"].fsm(state["threshold"])
        return dict(counts=r["counts"], sums=r["sums"], support=np.array([c[2] for c in r["candidates"]]),
                    labels=np.array([c[1] for c in r["candidates"]]))
    if kind == "paged":
        return state["g"].count_cliques(state["k"])
    if kind == "setops":
        r = kz.set_op_batch(state["op"], state["lists"], state["pairs"])
        if state["op"] == "intersect_count":
            return r
        values = np.zeros(state["ids"], np.uint32)  # the results one after another
        lengths = np.array([len(x) for x in r])
        np.concatenate(r, out=values[:lengths.sum()])
        return dict(values=values, lengths=lengths)
    srv = state["server"]
    tickets = [srv.submit(g, what, k or 4) for g, what, k in state["queries"]]
    return np.array([srv.poll(t, wait=True)["counts"] for t in tickets], dtype=np.uint64)


def _draws(case):
    """(vertices, edge draws) of a case's graph."""
    if case["family"] == "rmat":
        return 1 << case["scale"], case["ef"] << case["scale"]
    return case["n"], case["draws"]


def work(case):
    """The graph (8-byte row offsets, 4-byte ids; both directions where it is
    symmetric) or the set operations' lists read once; one operation per id."""
    kind = case["kind"]
    if kind == "setops":
        ids = case["pairs"] * case["longest"] / math.log(case["longest"])  # mean length of log-uniform lists
        return {"bytes": int(12 * ids), "flops": int(2 * ids)}
    if kind in ("batch", "serve"):
        # pool graphs: 2^17 vertices and 17 edges a vertex on average
        graphs = case["graphs"] if kind == "batch" else case["pool"] * 3
        n, m = graphs << 17, graphs * 17 << 17
        if kind == "serve":
            n, m = n + (1 << case["scale"]), m + (16 << case["scale"])
    else:
        n, m = _draws(case)
        if case["sym"]:
            m *= 2
    return {"bytes": 8 * n + 4 * m, "flops": m}


def exact(case, seed):
    """Every output is a whole number, compared as it is."""
    return None
