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


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_size3_plans_equal_the_interpreter_and_the_executor(kzdev, monkeypatch, name):
    kz = kzdev
    g = GRAPHS[name](kz)
    dg = g.to_device()
    rng = np.random.default_rng(len(name))
    for i in range(30):
        p = _plan(rng, outside=i % 5 == 4)
        print(f"[case] plan3 {name} {i}", flush=True)
        want = oracle.run_plan(p, g.rowptr, g.col)
        assert dg.count_plan(p) == want, (name, i)
        monkeypatch.setenv("KZ_PLAN_FLAT", "0")
        assert dg.count_plan(p) == want, (name, i)
        monkeypatch.delenv("KZ_PLAN_FLAT")
    dg.release()
