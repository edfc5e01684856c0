"""GPU tests of the serving loop (blpg_server_*): single LPs of mixed shapes in, results
equal to the batch solver's (same kernels, replayed from each shape's captured graph),
admission against the HBM budget, and a Poisson replay with latency statistics."""
import ctypes as C

import numpy as np
import pytest

import simplexprojects_amd as sa

pytestmark = pytest.mark.gpu

SHAPES5 = [(27, 32), (50, 48), (74, 83), (105, 103), (205, 203)]


def c5(i, count, first=0):
    m, n = SHAPES5[i]
    return sa.gen_config(5, 5, m, n, count, shape_idx=i, first=first, batch_count=1024)


def mixed(counts):
    lps = []
    for i, k in enumerate(counts):
        lps += c5(i, k)
    order = np.random.default_rng(0).permutation(len(lps))
    return [lps[k] for k in order]


def test_server_results_match_batch_solver():
    lps = mixed([40, 40, 40, 40, 8])
    S = sa.Solver(precision="fp64")
    ref = S.solve(lps)
    srv = sa.Server(S, max_batch=64, max_wait_us=100, precision="fp64")
    tickets = [srv.submit(lp, want_x=True) for lp in lps]
    got = {}
    while len(got) < len(lps):
        for r in srv.poll(wait_us=100000):
            got[r["ticket"]] = r
    for k, t in enumerate(tickets):
        r = got[t]
        assert r["status"] == ref.status[k] and r["pivots"] == ref.pivots[k]
        assert r["objective"] == ref.objective[k]
        assert np.array_equal(r["x"], ref.x[k]) and np.array_equal(r["basis"], ref.basis[k])
        assert r["latency_us"] > 0
    st = srv.stats()
    assert st["completed"] == len(lps) and st["batches"] >= 5 and st["rejected"] == 0
    srv.close()
    S.close()


def test_server_admission_budget():
    S = sa.Solver()
    srv = sa.Server(S, hbm_budget=1 << 20, max_batch=64)
    with pytest.raises(sa.BlpgError) as e:
        srv.submit(c5(3, 1)[0])
    assert e.value.code == sa.E_BUDGET
    assert srv.stats()["rejected"] == 1
    srv.close()
    S.close()


def test_server_poisson_replay():
    lps = mixed([200, 200, 200, 200, 40])
    rng = np.random.default_rng(1)
    arrival = np.cumsum(rng.exponential(1e6 / 20000.0, len(lps)))  # 20k LPs/s
    S = sa.Solver(precision="fp32")
    ref = sa.Solver(precision="fp64").solve(lps)
    srv = sa.Server(S, max_batch=256, max_wait_us=200, precision="fp32")
    res = srv.replay(lps, arrival)
    assert np.array_equal(res["status"], ref.status)
    opt = ref.status == sa.OPTIMAL
    rel = np.abs(res["objective"][opt] - ref.objective[opt]) / np.maximum(1, np.abs(ref.objective[opt]))
    assert rel.max() <= 1e-6
    st = srv.stats()
    assert st["completed"] == len(lps) and 0 < st["p50_us"] <= st["p99_us"] <= st["max_us"]
    assert (res["latency_us"] > 0).all()
    srv.close()
    S.close()


def test_server_burst_launches_every_full_arena():
    # Back-to-back submissions into arenas of 8 slots: an arena fills up and the next request
    # opens another arena of the shape before the worker has launched the full one.  The
    # worker launches every arena that holds requests, so all of them complete and match
    # the batch solver (regression: a full arena the filling had moved on from was never
    # launched, and its requests waited until the replay's stall report).
    lps = mixed([320, 320, 320, 320])
    ref = sa.Solver(precision="fp64").solve(lps)
    S = sa.Solver(precision="fp64")
    srv = sa.Server(S, max_batch=8, max_wait_us=1000, precision="fp64")
    for rnd in range(3):
        res = srv.replay(lps, np.zeros(len(lps)))
        assert np.array_equal(res["status"], ref.status), rnd
        assert np.array_equal(res["pivots"], ref.pivots), rnd
    assert srv.stats()["completed"] == 3 * len(lps)
    srv.close()
    S.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_server_tagged_warmstart_50k(precision):
    """The serving workload at its offered rate (Poisson 50k LPs/s, the five shapes, 64 GB
    budget) with a share of 105x103 requests tagged to known parametric families: every
    result is checked against the oracle; untagged FP64 results take the oracle's pivots,
    tagged ones are crashed from the trained network and take fewer pivots
    than the oracle's cold solves of the same LPs."""
    import oracle
    nf, m, n = 8, 105, 103
    train, tagged = [], []
    for f in range(nf):
        train += sa.gen_config(4, 7, m, n, 256, shape_idx=f, first=0, batch_count=1024)
        tagged += sa.gen_config(4, 7, m, n, 96, shape_idx=f, first=256, batch_count=1024)
    S = sa.Solver(precision="fp64")
    labels = S.solve(train)
    ws = sa.WarmStart(S, nf, m, n, seed=7, steps=400, lr=3e-3, weight_decay=1e-2)
    ws.train(train, labels.basis)
    lps = mixed([1200, 1200, 1200, 1200, 200]) + tagged
    lps = [lps[k] for k in np.random.default_rng(2).permutation(len(lps))]
    rng = np.random.default_rng(3)
    arrival = np.cumsum(rng.exponential(1e6 / 50000.0, len(lps)))
    Sp = sa.Solver(precision=precision)
    srv = sa.Server(Sp, max_batch=512, max_wait_us=200, precision=precision)
    srv.set_warmstart(ws)
    res = srv.replay(lps, arrival)
    st = srv.stats()
    srv.close()
    ref = oracle.solve_batch(lps, threads=8)
    is_tag = np.array([lp.family >= 0 for lp in lps])
    assert is_tag.sum() == nf * 96 and st["completed"] == len(lps) and st["rejected"] == 0
    assert np.array_equal(res["status"], ref["status"])
    opt = ref["status"] == sa.OPTIMAL
    rel = np.abs(res["objective"] - ref["objective"]) / np.maximum(1, np.abs(ref["objective"]))
    assert rel[opt].max() <= (1e-9 if precision == "fp64" else 1e-6)
    if precision == "fp64":
        # (objectives come from the FP64 check's refined solve: within 1e-9, not bitwise)
        plain = ~is_tag
        assert np.array_equal(res["pivots"][plain], ref["pivots"][plain])
    warm_piv = res["pivots"][is_tag].mean()
    cold_piv = ref["pivots"][is_tag].mean()
    assert warm_piv < 0.9 * cold_piv, (warm_piv, cold_piv)
    assert 0 < st["p50_us"] <= st["p99_us"]
    ws.close()
    Sp.close()
    S.close()


@pytest.mark.parametrize("precision,shape,want", [
    ("fp64", (105, 103), (sa.KERNEL_TILE, 4)), ("fp64", (174, 142), (sa.KERNEL_TILE, 5)),
    ("fp32", (174, 142), (sa.KERNEL_WAVE, 5)), ("fp32", (205, 203), (sa.KERNEL_WAVE, 6))])
def test_arena_instance_goes_by_size(precision, shape, want):
    """An arena's slots are a capacity, of which a launch usually fills a few: it takes the
    instance of its shape, not the one for as many LPs as it has slots."""
    info_of = getattr(sa.load_library(), "_ZN4blpg17server_arena_infoEP11blpg_serveriiP15blpg_batch_info")
    lp = sa.gen_config(2, 7, *shape, 1, batch_count=1)[0]
    S = sa.Solver(precision=precision)
    srv = sa.Server(S, max_batch=1024, arenas=1, precision=precision)
    srv.submit(lp)
    got = []
    while not got:
        got = srv.poll(wait_us=100000)
    info = sa._Info()
    assert info_of(srv.h, C.c_int(shape[0]), C.c_int(shape[1]), C.byref(info)) == 0
    assert (info.nbins, info.count[0]) == (1, 1024)
    assert (info.kernel[0], info.param[0]) == want
    assert got[0]["status"] == S.solve([lp]).status[0]
    srv.close()
    S.close()
