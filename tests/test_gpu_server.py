"""GPU tests of the query server (kz_server_*): every query in a mixed,
concurrently running stream returns the same exact count as the oracle
(alone-vs-mix parity), under no budget, under a budget that forces prepared
executions to be evicted and re-prepared, and with a budget too small for
any query (KZ_ERR_BUDGET)."""

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

APP = {3: "kautomine_triangle", 4: "kautomine_four_clique", 5: "kautomine_five_clique"}


def _pool(kz):
    sym = {
        "chunglu": kz.gen_chung_lu(6000, 30000, 2.3, 400, 3),
        "rmat11": kz.gen_rmat(11, 12, seed=9),
    }
    ori = {
        "rmat12_o": kz.gen_rmat(12, 16, seed=4).oriented(),
        "er_o": kz.gen_erdos_renyi(3000, 45000, 6).oriented(),
        "chunglu_o": sym["chunglu"].oriented(),
    }
    return sym, ori


def _expected(sym, ori):
    want = {}
    for name, g in ori.items():
        for k in (3, 4, 5):
            want[(name, "clique", k)] = [oracle.run_app(APP[k], g.rowptr, g.col)[1][0]]
    for name, g in sym.items():
        want[(name, "census", 0)] = oracle.motif_census(g.rowptr, g.col)
        want[(name, "clique", 4)] = [oracle.run_app(APP[4], g.rowptr, g.col)[1][0]]
    return want


def _run_stream(kz, server, dgs, queries):
    tickets = [(key, server.submit(dgs[key[0]], key[1], key[2] or 4)) for key in queries]
    out = []
    for key, t in tickets:
        res = server.poll(t, wait=True)
        out.append((key, res))
    return out


def test_server_mixed_stream_exact(kzdev):
    kz = kzdev
    sym, ori = _pool(kz)
    want = _expected(sym, ori)
    dgs = {name: g.to_device() for name, g in {**sym, **ori}.items()}
    keys = sorted(want)
    rng = np.random.default_rng(5)
    queries = [keys[i] for i in rng.integers(0, len(keys), 60)]
    print(f"[case] server mixed stream, {len(queries)} queries over {len(keys)} kinds", flush=True)
    with kz.Server(hbm_budget=0, max_inflight=4) as srv:
        for key, res in _run_stream(kz, srv, dgs, queries):
            assert res["status"] == 0, (key, res)
            n = len(want[key])
            assert res["counts"][:n] == want[key], (key, res["counts"], want[key])
            assert res["total_ms"] >= res["run_ms"] >= 0
        # non-blocking poll eventually returns the result
        t = srv.submit(dgs["rmat12_o"], "clique", 4)
        res = None
        while res is None:
            res = srv.poll(t)
        assert res["counts"][0] == want[("rmat12_o", "clique", 4)][0]
        with pytest.raises(kz.KzError):
            srv.poll(t)  # retired


def test_server_budget_eviction_and_rejection(kzdev):
    kz = kzdev
    sym, ori = _pool(kz)
    want = _expected(sym, ori)
    dgs = {name: g.to_device() for name, g in {**sym, **ori}.items()}
    keys = [k for k in sorted(want) if k[1] == "clique"]
    # room for roughly one prepared clique execution at a time: every switch
    # of (graph, k) evicts the previous one, counts must stay exact
    budget = 8 * 6000 + (1 << 20) + 8 * 6001 + 4 * (2 * 30000 + 8)
    print(f"[case] server eviction, budget {budget}", flush=True)
    with kz.Server(hbm_budget=budget * 3, max_inflight=2) as srv:
        for key, res in _run_stream(kz, srv, dgs, keys * 2):
            assert res["status"] == 0, (key, res)
            assert res["counts"][0] == want[key][0], key
    print("[case] server rejection", flush=True)
    with kz.Server(hbm_budget=4096, max_inflight=2) as srv:
        for key, res in _run_stream(kz, srv, dgs, keys[:3] + [("chunglu", "census", 0)]):
            assert res["status"] == kz._ffi.KZ_ERR_BUDGET, (key, res)


def test_queries_are_admitted_during_a_census_and_a_preparation(kzdev):
    """A census runs on a helper thread, and a clique job is prepared on
    another: a small clique query submitted behind either is admitted,
    launched and finished while they are still running, and every result
    stays exact."""
    kz = kzdev
    big_sym = kz.gen_chung_lu(1500000, 12000000, 2.3, 8000, 7)
    big_ori = kz.gen_rmat(21, 16, seed=3).oriented()
    small = kz.gen_rmat(12, 16, seed=4).oriented()
    want_small = oracle.run_app(APP[4], small.rowptr, small.col)[1][0]
    want_census = oracle.motif_census(big_sym.rowptr, big_sym.col)
    want_big = oracle.run_app(APP[3], big_ori.rowptr, big_ori.col)[1][0]
    d_sym, d_ori, d_small = big_sym.to_device(), big_ori.to_device(), small.to_device()
    with kz.Server(hbm_budget=0, max_inflight=4) as srv:
        # the small query's execution is prepared before the timed part
        assert srv.poll(srv.submit(d_small, "clique", 4), wait=True)["counts"][0] == want_small
        print("[case] clique query behind a census", flush=True)
        tc = srv.submit(d_sym, "census", 0)
        tq = srv.submit(d_small, "clique", 4)
        rq = srv.poll(tq, wait=True)
        census_running = srv.poll(tc) is None
        rc = srv.poll(tc, wait=True)
        assert rq["status"] == 0 and rq["counts"][0] == want_small
        assert rc["status"] == 0 and rc["counts"] == want_census
        assert census_running, (rq, rc)
        print("[case] clique query behind a preparation", flush=True)
        tb = srv.submit(d_ori, "clique", 3)
        tq = srv.submit(d_small, "clique", 4)
        rq = srv.poll(tq, wait=True)
        big_running = srv.poll(tb) is None
        rb = srv.poll(tb, wait=True)
        assert rq["status"] == 0 and rq["counts"][0] == want_small
        assert rb["status"] == 0 and rb["counts"][0] == want_big
        assert big_running, (rq, rb)


def _big_chunglu(kz):
    return kz.gen_chung_lu(20000, 400000, 2.2, 2000, 12)


def test_a_kept_job_whose_core_does_not_fit_beside_the_forward_copy(kzdev):
    """A symmetric graph counted directly first keeps its forward copy and a
    4-clique job with a core bitmap.  A budget that holds both without the
    bitmap serves the query, one that holds the bitmap too adopts the job."""
    kz = kzdev
    g = _big_chunglu(kz)
    want = oracle.run_app(APP[4], g.rowptr, g.col)[1][0]
    for slack, core_kept in ((0, True), (-1, False)):
        dg = g.to_device()
        assert dg.count_cliques(4) == want
        kept = dg.clique_kept_bytes(4)
        assert kept["forward"] and kept["core"] and kept["execution"] > kept["core"], kept
        budget = kept["forward"] + kept["execution"] + slack
        print(f"[case] server budget {budget} on {kept}", flush=True)
        with kz.Server(hbm_budget=budget, max_inflight=2) as srv:
            for _ in range(2):
                res = srv.poll(srv.submit(dg, "clique", 4), wait=True)
                assert res["status"] == 0 and res["counts"][0] == want, res
            now = dg.clique_kept_bytes(4)  # no query in flight
            assert now["core"] == (kept["core"] if core_kept else 0), now
        # without the bitmap it does not fit either: refused as before
        if not core_kept:
            dg2 = g.to_device()
            assert dg2.count_cliques(4) == want
            with kz.Server(hbm_budget=kept["forward"] + kept["execution"] - kept["core"] - 1, max_inflight=2) as srv:
                res = srv.poll(srv.submit(dg2, "clique", 4), wait=True)
                assert res["status"] == kz._ffi.KZ_ERR_BUDGET, res
            dg2.release()
        dg.release()


def test_a_core_bitmap_evicts_no_prepared_execution(kzdev):
    """Room for two executions but not for the second one's core bitmap: the
    first one stays prepared and the second runs without a bitmap."""
    kz = kzdev
    a, b = kz.gen_rmat(12, 16, seed=4).oriented(), _big_chunglu(kz).oriented()
    wa = oracle.run_app(APP[4], a.rowptr, a.col)[1][0]
    wb = oracle.run_app(APP[4], b.rowptr, b.col)[1][0]
    kept = {}
    for name, g, want in (("a", a, wa), ("b", b, wb)):
        probe = g.to_device()
        assert probe.count_cliques(4) == want
        kept[name] = probe.clique_kept_bytes(4)
        probe.release()
    assert kept["a"]["core"] and kept["b"]["core"], kept
    # an execution on an oriented graph without hubs is admitted at 8 bytes a
    # vertex and 1 MB, then held at its real size
    assert max(a.max_degree, b.max_degree) <= 1024
    budget = 8 * b.num_vertices + (1 << 20) + kept["b"]["core"] + kept["a"]["execution"] // 2
    assert kept["a"]["execution"] // 2 < kept["b"]["core"], kept
    da, db = a.to_device(), b.to_device()
    print(f"[case] server cores {kept}, budget {budget}", flush=True)
    with kz.Server(hbm_budget=budget, max_inflight=2) as srv:
        ra = srv.poll(srv.submit(da, "clique", 4), wait=True)
        rb = srv.poll(srv.submit(db, "clique", 4), wait=True)
        assert ra["counts"][0] == wa and rb["counts"][0] == wb, (ra, rb)
        now = da.clique_kept_bytes(4), db.clique_kept_bytes(4)  # no query in flight
    assert now[0] == kept["a"], "the first execution was released or lost its bitmap"
    assert now[1]["execution"] and now[1]["core"] == 0, now
    da.release()
    db.release()


def test_a_census_whose_optional_parts_do_not_fit(kzdev, monkeypatch):
    """The census copy's core bitmap and range histograms are left out where
    the budget has no room for them, in a copy kept from a direct call and in
    one that the server builds; the copy then stays with the server."""
    kz = kzdev
    monkeypatch.setenv("KZ_C4_RANGE_BOUND", "4096")  # histograms at this size
    monkeypatch.setenv("KZ_C4_SCRATCH_KEYS", "9000")  # a scratch below the server's estimate
    g = kz.gen_chung_lu(300000, 1500000, 2.2, 5000, 21)
    want = oracle.motif_census(g.rowptr, g.col)
    dg = g.to_device()
    assert dg.motif_census() == want
    full = dg.census_kept_bytes()
    dg.release()
    assert full["extra"] > 1 << 20, full
    cases = [  # budget, counted directly before, optional bytes kept
        (full["state"], True, full["extra"]),
        (full["state"] - 1, True, 0),
        (full["state"] - full["extra"], True, 0),
        (0, False, full["extra"]),
    ]
    for budget, direct, extra in cases:
        dg = g.to_device()
        if direct:
            assert dg.motif_census() == want
        print(f"[case] server census, budget {budget}, kept {direct}, of {full}", flush=True)
        with kz.Server(hbm_budget=budget, max_inflight=2) as srv:
            for _ in range(2):
                res = srv.poll(srv.submit(dg, "census", 0), wait=True)
                assert res["status"] == 0 and res["counts"] == want, res
                now = dg.census_kept_bytes()  # no query in flight
                assert now["state"] - now["extra"] == full["state"] - full["extra"], (now, full)
                assert now["extra"] == extra, (now, full)
        dg.release()
    # a budget for the server's own upper estimate alone: no optional part
    n, m = g.num_vertices, g.num_entries
    col = 4 * ((m + 3) // 4 * 4 + 4)
    cus = kz.device_info()["compute_units"]
    need = 8 * (n + 1) * 3 + 3 * col + 16 * n * cus + 8 * n + (1 << 20)
    for budget, extra in ((need, False), (need - 1, None)):
        dg = g.to_device()
        print(f"[case] server census, budget {budget}", flush=True)
        with kz.Server(hbm_budget=budget, max_inflight=2) as srv:
            res = srv.poll(srv.submit(dg, "census", 0), wait=True)
            if extra is None:
                assert res["status"] == kz._ffi.KZ_ERR_BUDGET, res
            else:
                assert res["status"] == 0 and res["counts"] == want, res
                now = dg.census_kept_bytes()
                assert now["state"] and now["extra"] == 0, now
        dg.release()
