"""GPU parity of the induced 3-/4-vertex motif census (kz_motif_census)
against the oracle: exhaustive enumeration on small graphs, the
combinatorial oracle on larger ones, and the three_motif apps' own counts
for the 3-vertex part (kautomine/three_motif.cc)."""

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def test_census_small_graphs_brute_force(kzdev):
    kz = kzdev
    rng = np.random.default_rng(11)
    for case in range(40):
        n = int(rng.integers(4, 60))
        m = int(rng.integers(1, n * (n - 1) // 2 + 1))
        s, t = rng.integers(0, n, m), rng.integers(0, n, m)
        g = kz.from_edges(np.concatenate([s, t]), np.concatenate([t, s]), n)
        if g.num_vertices == 0:
            continue
        print(f"[case] small census #{case} n={g.num_vertices} entries={g.num_entries}", flush=True)
        want = oracle.brute_motifs(g.rowptr, g.col)
        dg = g.to_device()
        assert dg.motif_census() == want, case
        dg.release()


def _medium(kz):
    yield "chunglu_20k", kz.gen_chung_lu(20000, 120000, 2.3, 2000, 7)
    yield "rmat13", kz.gen_rmat(13, 16, seed=4)
    yield "er_4k", kz.gen_erdos_renyi(4000, 60000, 3)
    yield "dense_er", kz.gen_erdos_renyi(400, 40000, 8)


@pytest.mark.parametrize("name", ["chunglu_20k", "rmat13", "er_4k", "dense_er"])
def test_census_matches_oracle(kzdev, name):
    kz = kzdev
    g = dict(_medium(kz))[name]
    print(f"[case] census {name} n={g.num_vertices} entries={g.num_entries}", flush=True)
    want = oracle.motif_census(g.rowptr, g.col)
    dg = g.to_device()
    got = dg.motif_census()
    assert got == want, (name, got, want)
    # repeated calls reuse the relabelled copy and must agree
    assert dg.motif_census() == want
    # the 3-vertex part is what the kautomine three_motif app prints, in its
    # pattern order (triangle, wedge)
    assert oracle.run_app("kautomine_three_motif", g.rowptr, g.col)[1] == [want[1], want[0]]
    dg.release()


@pytest.mark.parametrize("scratch,slots,direct", [("3000", None, "0"), ("500", None, "0"), (None, "64", None),
                                                  ("700", "128", "0"), (None, None, "0"), ("20000", "256", "2000")])
def test_census_heavy_root_paths(kzdev, monkeypatch, scratch, slots, direct):
    """Roots above the workgroup hash first try one pass over the LDS table
    (direct); the others bucket their wedge endpoints through an HBM scratch
    region.  A small region makes them take several rounds and fill buckets
    (the exact path), and buckets larger than the region are counted from
    the wedge stream.  A small table makes the counts split buckets into
    parts and makes direct attempts fail."""
    kz = kzdev
    knobs = {"KZ_C4_SCRATCH_KEYS": scratch, "KZ_C4_BUCKET_SLOTS": slots, "KZ_C4_DIRECT_BOUND": direct}
    for name in ("dense_er", "chunglu_20k", "rmat13"):
        g = dict(_medium(kz))[name]
        want = oracle.motif_census(g.rowptr, g.col)
        for k, v in knobs.items():
            if v is not None:
                monkeypatch.setenv(k, v)
        print(f"[case] census {name} {knobs}", flush=True)
        dg = g.to_device()  # the settings are read when the census state is built
        got = dg.motif_census()
        dg.release()
        for k in knobs:
            monkeypatch.delenv(k, raising=False)
        assert got == want, (name, knobs)


def test_census_rejects_oriented_graph(kzdev):
    kz = kzdev
    dg = kz.gen_erdos_renyi(500, 3000, 1).oriented().to_device()
    with pytest.raises(kz.KzError):
        dg.motif_census()
    dg.release()


@pytest.mark.parametrize("n,knobs", [
    (25000, {}), (60000, {}),  # counters of every id: one range, two
    (66000, {}), (150000, {}), (400000, {}),  # more ranges: bucketed by range above the default bound
    (400000, {"KZ_C4_RANGE_BOUND": "4096"}),
    (400000, {"KZ_C4_RANGE_BOUND": "4096", "KZ_C4_SCRATCH_KEYS": "9000"}),  # rounds of ranges
    (400000, {"KZ_C4_RANGE_BOUND": "4096", "KZ_C4_SCRATCH_KEYS": "300"}),  # ranges above the scratch
])
def test_census_direct_counters(kzdev, monkeypatch, n, knobs):
    """Heavy roots counted in one counter per id, by range."""
    kz = kzdev
    g = kz.gen_chung_lu(n, 5 * n, 2.2, 6000, n)
    want = oracle.motif_census(g.rowptr, g.col)
    for k, v in knobs.items():
        monkeypatch.setenv(k, v)
    print(f"[case] census n={n} {knobs}", flush=True)
    dg = g.to_device()
    got = dg.motif_census()
    again = dg.motif_census()
    dg.release()
    assert got == want and again == want


def test_census_counts_above_16_bits(kzdev):
    """Two vertices with 70,000 common neighbours: one counter reaches 70,000,
    in a graph that is bucketed by range."""
    kz = kzdev
    k = 70000
    leaves = np.arange(2, k + 2, dtype=np.uint32)
    g = kz.from_edges(np.repeat(np.array([0, 1], np.uint32), k), np.concatenate([leaves, leaves]), k + 2)
    print(f"[case] census K(2,{k})", flush=True)
    dg = g.to_device()
    got = dg.motif_census()
    dg.release()
    # induced: wedges (two leaves at a hub, the hubs at a leaf), no 3-path
    # (hub - leaf - hub - leaf closes a 4-cycle), stars of three leaves
    assert got == [k * (k - 1) + k, 0, 0, k * (k - 1) * (k - 2) // 3, k * (k - 1) // 2, 0, 0, 0]
