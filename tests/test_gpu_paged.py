"""Graphs beyond HBM (kz_paged_*): the neighbour lists stay in pinned host
memory and each batch of roots fetches what it needs through a device-side
deduplicated request list and an HBM cache of high-degree lists (the remote
graph-data path of src/engine.cc:94-510).  With a working budget forced far
below the graph's size, every count must equal the oracle's and the resident
form's, for any cache size; requests must be deduplicated and every fetched
byte accounted to the cache or to host memory."""

import pytest

import oracle

pytestmark = pytest.mark.gpu

APPS = {3: "kautomine_triangle", 4: "kautomine_four_clique", 5: "kautomine_five_clique"}


def _graphs(kz):
    return [("rmat15", kz.gen_rmat(15, 16, seed=4).oriented()),
            ("chunglu", kz.gen_chung_lu(40000, 300000, 2.3, 4000, 8).oriented()),
            ("er", kz.gen_erdos_renyi(20000, 200000, 5).oriented())]


@pytest.mark.parametrize("cache", [0, 1 << 20, 1 << 30])
def test_paged_counts_equal_the_oracle(kzdev, cache):
    kz = kzdev
    for name, g in _graphs(kz):
        lists = 4 * g.num_entries
        budget = max(lists // 8, 1 << 16)
        print(f"[case] paged {name} list_bytes={budget} cache={cache}", flush=True)
        # the largest cache takes every list (threshold 1), the others the
        # lists of vertices of total degree >= 32
        pg = kz.PagedGraph(g, list_bytes=budget, cache_bytes=cache,
                           cache_degree_threshold=1 if cache >= lists else 32)
        dg = g.to_device()
        for k in (3, 4, 5):
            want = oracle.run_app(APPS[k], g.rowptr, g.col)[1][0]
            got = pg.count_cliques(k)
            st = pg.last_stats
            assert got == want, (name, k, cache)
            assert dg.count_cliques(k) == want
            assert st["batches"] >= 2, st
            assert st["requests"] < st["request_refs"], st  # deduplicated
            if cache == 0:
                assert st["cache_bytes"] == 0 and st["cached_vertices"] == 0
            if cache >= lists:
                assert st["host_bytes"] == 0, st
        pg.release()
        dg.release()


def test_paged_counts_of_a_graph_cut_in_pieces(kzdev):
    """More than one piece of roots: the counted batches are the cut's."""
    import ctypes as C

    from openkhuzdulgraph_amd import _ffi
    kz = kzdev
    g = kz.gen_rmat(18, 10, seed=3).oriented()
    want = oracle.run_app(APPS[3], g.rowptr, g.col)[1][0]
    print("[case] paged pieces", flush=True)
    assert g.num_entries > 2 << 20  # two pieces
    nb = C.c_uint32()
    assert _ffi.lib().kz_paged_plan(C.byref(g._raw), g.num_entries, 0, None, None, C.byref(nb)) == 0
    pg = kz.PagedGraph(g, list_bytes=g.num_entries, cache_bytes=0)
    assert pg.count_cliques(3) == want
    assert pg.last_stats["batches"] == nb.value
    pg.release()


def test_paged_refuses_a_budget_below_one_root(kzdev):
    kz = kzdev
    g = kz.gen_rmat(12, 16, seed=2).oriented()
    with pytest.raises(kz.KzError) as ei:
        kz.PagedGraph(g, list_bytes=64)
    from openkhuzdulgraph_amd import _ffi
    assert ei.value.code == _ffi.KZ_ERR_BUDGET


def test_unchanged_apps_beyond_the_resident_budget(kzdev, tmp_path):
    """KZ_RESIDENT_BYTES below the graph's lists: the unchanged clique apps
    run on the paged form (cache_degree_threshold and relative_cache_size
    of the app's DistributedApplication size the cache) and print the
    reference binaries' counts (symmetric RMAT-16, oriented on the host)."""
    import json
    import os
    import re
    import subprocess
    from pathlib import Path

    from openkhuzdulgraph_amd import workloads as wl
    root = Path(__file__).resolve().parent.parent
    apps = root / "openkhuzdulgraph_amd" / "khuzdul" / "_apps"
    if not apps.is_dir():
        pytest.skip("app binaries were not built from the reference sources")
    gold = json.loads((root / "tests" / "golden" / "config_counts.json").read_text())["sym_rmat16_ef16"]
    g = wl.rmat(kzdev, 16, 16, orient=False)
    assert f"{g.digest():016x}" == gold["digest"]
    path = tmp_path / "rmat16_sym.dgraph"
    g.store(str(path))
    env = dict(os.environ, KZ_RESIDENT_BYTES=str(1 << 20))
    for app in ("kautomine_four_clique", "kgraphpi_triangle"):
        print(f"[case] paged app={app}", flush=True)
        out = subprocess.run([str(apps / app), str(path), "1", "1"], env=env, capture_output=True, text=True,
                             timeout=300)
        assert out.returncode == 0, out.stderr[-2000:]
        assert "stay in host memory" in out.stdout
        got = {int(m.group(1)): int(m.group(2)) for m in re.finditer(r"Pattern count (\d+): (\d+)", out.stdout)}
        assert got.get(0) == gold["counts"][f"reference:{app}"], out.stdout[-1500:]
