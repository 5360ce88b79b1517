"""Counting plans of pattern size 3: the closed form against the oracle's plan
interpreter and the level-by-level executor (KZ_PLAN_FLAT=0), over random
plans of the accepted form and plans and graphs just outside it."""

import numpy as np
import pytest

import oracle
from openkhuzdulgraph_amd import _ffi

pytestmark = pytest.mark.gpu


def _plan(rng, outside=False):
    """Random size-3 plan: scatters and counts of N(v0) at size 1; up to three
    operations on N(v0), N(v1) and counts of them or of the lists at size 2."""
    p = _ffi.kz_plan_desc()
    p.pattern_size = 3
    p.num_aggregators = 3
    p.num_step_lists = 4
    for s in range(_ffi.KZ_MAX_PATTERN):
        for c in range(256):
            p.type_table[s][c] = 0xFF

    def ref(r, kind, a, b=0):
        r.kind, r.a, r.b = kind, a, b

    root = p.lists[0]
    root.num_ops, root.num_outs = 0, int(rng.integers(1, 3))
    for o in range(root.num_outs):
        out = root.outs[o]
        out.kind = _ffi.KZ_OUT_SCATTER if o == 0 else int(rng.choice([_ffi.KZ_OUT_SCATTER, _ffi.KZ_OUT_COUNT]))
        out.aggregator, out.pred = int(rng.integers(0, 3)), int(rng.integers(0, 8))
        ref(out.src, _ffi.KZ_SET_NBR, 0)
    p.type_table[1][0] = 0
    for code in range(3):
        p.type_table[2][code] = 1 + code
        lst = p.lists[1 + code]
        lst.num_ops, lst.num_outs = int(rng.integers(0, 4)), int(rng.integers(1, 5))
        for j in range(lst.num_ops):
            lst.ops[j].op = int(rng.choice([_ffi.KZ_OP_INTERSECT, _ffi.KZ_OP_SUBTRACT]))
            ref(lst.ops[j].lhs, _ffi.KZ_SET_NBR, int(rng.integers(0, 2)))
            ref(lst.ops[j].rhs, _ffi.KZ_SET_NBR, int(rng.integers(0, 2)))
            if outside and j:
                ref(lst.ops[j].lhs, _ffi.KZ_SET_SLOT, 2, j - 1)
        for o in range(lst.num_outs):
            out = lst.outs[o]
            out.kind, out.aggregator, out.pred = _ffi.KZ_OUT_COUNT, int(rng.integers(0, 3)), int(rng.integers(0, 32))
            if lst.num_ops and rng.random() < 0.7:
                ref(out.src, _ffi.KZ_SET_SLOT, 2, int(rng.integers(0, lst.num_ops)))
            else:
                ref(out.src, _ffi.KZ_SET_NBR, int(rng.integers(0, 2)))
    return p


def _one_way(kz):
    """A directed graph that is neither oriented nor symmetric, with a
    self-loop and a vertex without neighbours."""
    import tempfile

    pairs = np.array([[0, 1], [0, 2], [1, 0], [1, 2], [2, 2], [2, 3], [3, 0], [5, 1]], np.uint32)
    with tempfile.NamedTemporaryFile(suffix=".dgraph") as f:
        f.write(np.uint32(6).tobytes() + np.uint64(len(pairs)).tobytes() + np.zeros(2, np.int32).tobytes())
        f.write(pairs.tobytes())
        f.flush()
        return kz.load_dgraph(f.name)


def _two_cycles(kz):
    """As many entries below as above their vertices, but one way round."""
    import tempfile

    pairs = np.array([[0, 1], [1, 2], [2, 0], [3, 0]], np.uint32)
    with tempfile.NamedTemporaryFile(suffix=".dgraph") as f:
        f.write(np.uint32(4).tobytes() + np.uint64(len(pairs)).tobytes() + np.zeros(2, np.int32).tobytes())
        f.write(pairs.tobytes())
        f.flush()
        return kz.load_dgraph(f.name)


GRAPHS = {
    "rmat_sym": lambda kz: kz.gen_rmat(9, 12, seed=8),
    "rmat_oriented": lambda kz: kz.gen_rmat(9, 12, seed=8).oriented(),
    "chunglu_sym": lambda kz: kz.gen_chung_lu(1500, 9000, 2.2, 300, 4),
    "star": lambda kz: kz.from_edges(np.zeros(200, np.uint32), np.arange(1, 201, dtype=np.uint32), 201),
    "complete": lambda kz: kz.from_edges(*np.triu_indices(40, 1), 40),
    "one_way": _one_way,
    "two_cycles": _two_cycles,
}


QUALIFY = {"rmat_sym", "rmat_oriented", "chunglu_sym", "star", "complete"}  # no self-loop, upwards or both ways


def _closed(p, oriented):
    """Whether plan p has the closed form: the operations and counts of the
    order codes that its scatters reach, restated from the plan alone."""
    scatters = [p.lists[0].outs[o].pred for o in range(p.lists[0].num_outs)
                if p.lists[0].outs[o].kind == _ffi.KZ_OUT_SCATTER]
    reached = [c for c, bit in ((1, 0), (2, 2)) if any((s >> bit) & 1 for s in scatters)]
    for code in reached:
        if oriented and code == 1:
            continue
        lst = p.lists[p.type_table[2][code]]
        ops = [lst.ops[j] for j in range(lst.num_ops)]
        if any(r.kind != _ffi.KZ_SET_NBR for op in ops for r in (op.lhs, op.rhs)):
            return False
        for o in range(lst.num_outs):
            src = lst.outs[o].src
            if src.kind == _ffi.KZ_SET_NBR:
                whole = src.a
            else:
                op = ops[src.b]
                alone = op.lhs.a == op.rhs.a if op.op == _ffi.KZ_OP_INTERSECT else op.lhs.a != op.rhs.a
                whole = op.lhs.a if alone else None
            if oriented and whole == 1:
                return False
    return True


def _took_closed_form(stats):
    return stats["peak_bytes"] == 8 * 7 and stats["launches"] in (1, 2) and stats["chunks"] == 1


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_size3_plans_equal_the_interpreter_and_the_executor(kzdev, monkeypatch, name):
    kz = kzdev
    g = GRAPHS[name](kz)
    dg = g.to_device()
    rng = np.random.default_rng(len(name))
    taken = 0
    for i in range(30):
        p = _plan(rng, outside=i % 5 == 4)
        print(f"[case] plan3 {name} {i}", flush=True)
        want = oracle.run_plan(p, g.rowptr, g.col)
        assert dg.count_plan(p) == want, (name, i)
        closed = name in QUALIFY and _closed(p, g.oriented_flag)
        assert _took_closed_form(dg.last_stats) == closed, (name, i, dg.last_stats)
        taken += closed
        monkeypatch.setenv("KZ_PLAN_FLAT", "0")
        assert dg.count_plan(p) == want, (name, i)
        assert not _took_closed_form(dg.last_stats)
        monkeypatch.delenv("KZ_PLAN_FLAT")
    assert taken >= 5 if name in QUALIFY else taken == 0
    dg.release()


def test_threads_run_plans_and_counts_on_one_graph(kzdev):
    """Threads share a graph: the closed form's first calls (forward copy,
    3-clique execution) and later ones, beside clique counts of the same k and
    plans that take the executor, all at once."""
    import threading

    kz = kzdev
    g = kz.gen_rmat(12, 12, seed=5)
    rng = np.random.default_rng(3)
    plans = [_plan(rng, outside=i % 4 == 3) for i in range(8)]
    want = [oracle.run_plan(p, g.rowptr, g.col) for p in plans]
    tri = oracle.run_app("kautomine_triangle", g.rowptr, g.col)[1][0]
    assert sum(_closed(p, False) for p in plans) >= 4
    for _ in range(3):
        dg = g.to_device()
        print("[case] threads on one graph", flush=True)
        gate, bad = threading.Barrier(6), []

        def work(t):
            gate.wait()
            for i in range(8):
                j = (i + t) % 8
                got = dg.count_cliques(3) if t == 5 else dg.count_plan(plans[j])
                if got != (tri if t == 5 else want[j]):
                    bad.append((t, j, got))

        threads = [threading.Thread(target=work, args=(t,)) for t in range(6)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad, bad[:3]
        dg.release()


def test_roots_too_wide_for_the_triangle_count(kzdev):
    """An oriented graph with a root of 9,000 neighbours, more than the clique
    kernels take: plans that count common neighbours run on the executor, the
    others in closed form."""
    import tempfile

    kz = kzdev
    rng = np.random.default_rng(1)
    pairs = np.concatenate([np.stack([np.zeros(9000, np.int64), np.arange(1, 9001)], 1),
                            np.sort(rng.choice(9001, (3000, 2)), 1)])
    pairs = np.unique(pairs[pairs[:, 0] < pairs[:, 1]], axis=0).astype(np.uint32)
    with tempfile.NamedTemporaryFile(suffix=".dgraph") as f:
        f.write(np.uint32(9001).tobytes() + np.uint64(len(pairs)).tobytes() + np.zeros(2, np.int32).tobytes())
        f.write(pairs.tobytes())
        f.flush()
        g = kz.load_dgraph(f.name)
    assert g.oriented_flag and g.max_degree == 9000
    dg = g.to_device()
    seen = set()
    for i in range(24):
        p = _plan(rng)
        closed = _closed(p, True)
        # counts of a third corner above v0 < v1 (a plan whose operation is
        # the same on both lists counts none)
        reached = any((p.lists[0].outs[o].pred >> 2) & 1 for o in range(p.lists[0].num_outs)
                      if p.lists[0].outs[o].kind == _ffi.KZ_OUT_SCATTER)
        lst = p.lists[p.type_table[2][2]]
        common = [lst.ops[j].lhs.a != lst.ops[j].rhs.a for j in range(lst.num_ops)]
        members = reached and any(lst.outs[o].src.kind == _ffi.KZ_SET_SLOT and common[lst.outs[o].src.b]
                                  and (lst.outs[o].pred >> 4) & 1 for o in range(lst.num_outs))
        for _ in range(2):
            assert dg.count_plan(p) == oracle.run_plan(p, g.rowptr, g.col), i
            assert _took_closed_form(dg.last_stats) == (closed and not members), (i, dg.last_stats)
        seen.add((closed, members))
    assert {(True, True), (True, False)} <= seen
    dg.release()
