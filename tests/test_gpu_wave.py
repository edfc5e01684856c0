"""The matrix-core FP32 kernel at the edges of its tiles: row counts around multiples of 16,
column counts around multiples of 64, the smallest LP and each instance's full capacity,
through every stage (phase I, equality rows, degenerate rows, crash from a warm list).  The
arithmetic is the oracle's, so status, pivots, basis and the FP32 path are equal, bit for bit.
"""
import numpy as np
import pytest

import oracle
import simplexprojects_amd as sa

pytestmark = pytest.mark.gpu

# (variant, rows, columns): 16 chunks of rows and 64-column groups minus x0
EDGES = [(0, 1, 1), (0, 15, 63), (0, 16, 31), (0, 17, 62), (0, 32, 63), (1, 33, 63), (1, 64, 63),
         (2, 47, 64), (2, 64, 127), (3, 65, 65), (3, 80, 127), (4, 81, 126), (4, 112, 127),
         (5, 113, 128), (5, 176, 191), (6, 177, 192), (6, 208, 255), (7, 209, 255), (7, 256, 255)]


@pytest.mark.parametrize("variant,m,n", EDGES)
@pytest.mark.parametrize("cfg", [2, 3])
def test_tile_edges_vs_oracle(variant, m, n, cfg):
    count = 12 if m * n < 8192 else 4
    lps = sa.gen_config(cfg, 21, m, n, count, batch_count=count)
    S = sa.Solver(precision="fp32")
    S.tune_set(m, n, "wave", variant)
    r = S.solve(lps)
    for k, lp in enumerate(lps):
        if r.fallback[k]:
            continue  # re-solved in FP64
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision="fp32")
        assert r.status[k] == o["status"], k
        assert (r.pivots[k], r.phase1_pivots[k]) == (o["pivots"], o["phase1_pivots"]), k
        assert np.array_equal(r.basis[k], o["basis"]), k
    S.close()


@pytest.mark.parametrize("bland_after", [1, 2])
def test_bland_inside_a_run_of_pivots(bland_after):
    """Bland's rule sets in and goes out again between pivots of one run."""
    lps = sa.gen_config(2, 5, 40, 44, 24, batch_count=24)
    S = sa.Solver(precision="fp32", bland_after=bland_after)
    r = S.solve(lps)
    for k, lp in enumerate(lps):
        if not r.fallback[k]:
            o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision="fp32", bland_after=bland_after)
            assert (r.status[k], r.pivots[k]) == (o["status"], o["pivots"]), k
    S.close()


@pytest.mark.parametrize("max_iter", [1, 7])
def test_iteration_limit_inside_a_run(max_iter):
    lps = sa.gen_config(2, 5, 60, 80, 12, batch_count=12)
    S = sa.Solver(precision="fp32", max_iter=max_iter)
    r = S.solve(lps)
    for k, lp in enumerate(lps):
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision="fp32", max_iter=max_iter)
        if not r.fallback[k]:
            assert (r.status[k], r.pivots[k]) == (o["status"], o["pivots"]), k
    S.close()
