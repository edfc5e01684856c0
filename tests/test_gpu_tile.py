"""The 2-D block kernel at the edges of its blocks: the smallest LP, one row or column more
than a whole number of thread rows / columns, each variant's full capacity; cold and from a
warm list (block crash), through every stage, in both precisions.  Equal to the oracle's
replay: status, pivots and basis, and in FP64 objective and x, bit for bit.
"""
import numpy as np
import pytest

import oracle
import simplexprojects_amd as sa

pytestmark = pytest.mark.gpu

# variant: (thread rows, thread columns, rows, columns) of its capacity, objective rows,
# right-hand side and x0 included
CAPS = {0: (8, 8, 32, 40), 1: (8, 8, 56, 56), 2: (8, 16, 64, 112), 3: (8, 16, 80, 96),
        4: (16, 16, 112, 112), 5: (32, 16, 192, 144), 6: (32, 16, 224, 208),
        7: (8, 8, 80, 88), 8: (4, 16, 64, 112), 9: (8, 16, 112, 112), 10: (8, 32, 112, 128),
        11: (32, 16, 128, 112)}


def shapes(v):
    tr, tc, rows, cols = CAPS[v]
    return [(1, 1), (tr - 1, tc - 1), (2 * tr - 1, 2 * tc - 3), (rows - 2, cols - 2)]


@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("variant", sorted(CAPS))
def test_block_edges_vs_oracle(variant, precision, warm):
    for (m, n) in shapes(variant):
        for cfg in (2, 3):
            count = 6 if m * n < 8192 else 3
            lps = sa.gen_config(cfg, 31, m, n, count, batch_count=count)
            if warm:
                rng = np.random.default_rng(m * n)
                for lp in lps:
                    w = oracle.solve(lp.A, lp.b, lp.c, lp.sense)["basis"].copy()
                    w[w >= m + n] = -1
                    rng.shuffle(w)
                    w[rng.integers(m)] = rng.integers(n + m)  # possibly a wrong or repeated id
                    lp.warm_basis = w
            S = sa.Solver(precision=precision, verify=False)
            S.tune_set(m, n, "tile", variant)
            r = S.solve(lps)
            for k, lp in enumerate(lps):
                if r.fallback[k]:
                    continue  # an FP32 result re-solved in FP64
                o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision=precision,
                                 warm=lp.warm_basis)
                assert r.status[k] == o["status"], (m, n, cfg, k)
                assert (r.pivots[k], r.phase1_pivots[k]) == (o["pivots"], o["phase1_pivots"])
                assert np.array_equal(r.basis[k], o["basis"])
                if precision == "fp64":
                    assert r.objective[k] == o["objective"]
                    assert np.array_equal(r.x[k], o["x"])
            S.close()
