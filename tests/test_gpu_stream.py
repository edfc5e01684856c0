"""The HBM-streamed kernel: pending pivots applied to the slab in panels.  LPs whose pivot
counts end before, at and after a full panel, that replace the same row or column again
within a panel, larger than every register kernel holds, and with the vectors in HBM (beyond
LDS); every stage, cold and from a warm list.  Equal to the oracle's replay.
"""
import numpy as np
import pytest

import oracle
import simplexprojects_amd as sa

pytestmark = pytest.mark.gpu


def check(lps, precision, nt):
    m, n = lps[0].m, lps[0].n
    S = sa.Solver(precision=precision, verify=False)
    S.tune_set(m, n, "stream", nt)
    r = S.solve(lps)
    for k, lp in enumerate(lps):
        if r.fallback[k]:
            continue  # an FP32 result re-solved in FP64
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision=precision, warm=lp.warm_basis)
        assert r.status[k] == o["status"], k
        assert (r.pivots[k], r.phase1_pivots[k]) == (o["pivots"], o["phase1_pivots"]), k
        assert np.array_equal(r.basis[k], o["basis"]), k
        if precision == "fp64":
            assert r.objective[k] == o["objective"] and np.array_equal(r.x[k], o["x"]), k
    S.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nt", [64, 128, 256, 512])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 5), (9, 7), (40, 33), (65, 64)])
def test_small_panels(m, n, nt, precision):
    for cfg in (2, 3):
        check(sa.gen_config(cfg, 41, m, n, 10, batch_count=10), precision, nt)
    lps = sa.gen_config(3, 43, m, n, 6, batch_count=6)
    for lp in lps:  # crash from the optimal basis
        w = oracle.solve(lp.A, lp.b, lp.c, lp.sense)["basis"].copy()
        w[w >= m + n] = -1
        lp.warm_basis = w
    check(lps, precision, nt)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("m,n,cfg", [(260, 300, 2), (60, 1500, 2), (1200, 40, 1), (300, 260, 3),
                                     (20, 4000, 1), (4000, 20, 1), (1500, 1400, 1)])
def test_beyond_registers(m, n, cfg, precision):
    check(sa.gen_config(cfg, 47, m, n, 2, batch_count=2), precision, 512)


@pytest.mark.parametrize("max_iter", [1, 7, 8, 9, 16, 17])
def test_stop_within_a_panel(max_iter):
    lps = sa.gen_config(2, 51, 40, 50, 6, batch_count=6)
    S = sa.Solver(precision="fp64", verify=False, max_iter=max_iter, kernel="stream")
    r = S.solve(lps)
    for k, lp in enumerate(lps):
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, max_iter=max_iter)
        assert (r.status[k], r.pivots[k], r.objective[k]) == (o["status"], o["pivots"], o["objective"])
        assert np.array_equal(r.basis[k], o["basis"]) and np.array_equal(r.x[k], o["x"])
    S.close()
