"""GPU tests of infeasible LPs whose staged blocks are one column wider than min(m, n): phase
I ends with every structural and the auxiliary x0 basic, so the check stages n + 1 slack
columns.  Every such LP is checked and its own result reported, also where a check tier takes
a whole batch by itself, and in the host copy that the check of a later solve writes."""
import numpy as np
import pytest

import oracle
import simplexprojects_amd as sa

pytestmark = pytest.mark.gpu


def infeasible(m, n):
    """x_j <= 1, sum x >= n + (n + 1) / 2 and, up to m rows, x_1 <= 100: the phase-I optimum
    is x0 = 1/2, x_j = 3/2, so every x_j and x0 are basic."""
    A = np.zeros((m, n))
    b = np.full(m, 100.0)
    A[:, 0] = 1.0
    A[:n] = np.eye(n)
    b[:n] = 1.0
    A[n], b[n] = -1.0, -(n + (n + 1) / 2)
    return sa.LP(A, b, np.ones(n))


def feasible(m, n):
    return sa.LP(infeasible(m, n).A, np.full(m, 3.0), np.ones(n))


def overwrite(raw, lps):
    """Other values in the batch's host copy of the results."""
    k = len(lps)
    for f, size in (("status", k), ("pivots", k), ("phase1_pivots", k), ("fallback_used", k),
                    ("objective", k), ("kkt_primal", k), ("kkt_dual", k),
                    ("x", sum(lp.n for lp in lps)), ("basis", sum(lp.m for lp in lps))):
        np.ctypeslib.as_array(getattr(raw, f), shape=(size,))[:] = -77


# 2x1 .. 6x5: the tier's LDS is cut to the shape's own largest block; 60x35, 80x23 (first
# tier) and 78x75 (second tier): its LDS budget lies between n and n + 1 columns
@pytest.mark.parametrize("shape", [(2, 1), (4, 3), (6, 5), (60, 35), (80, 23), (78, 75)])
@pytest.mark.parametrize("count", [1, 300])
@pytest.mark.parametrize("graph", [False, True])
def test_infeasible_with_every_structural_basic(shape, count, graph):
    bad = infeasible(*shape)
    o = oracle.solve(bad.A, bad.b, bad.c, precision="fp32")
    assert o["status"] == oracle.INFEASIBLE
    assert set(range(shape[1])) <= set(o["basis"].tolist()) and sum(shape) in o["basis"]
    S = sa.Solver(precision="fp32", use_graph=graph)
    b = S.upload([feasible(*shape)] * count)
    b.solve()
    assert (b.fetch().status == oracle.OPTIMAL).all()
    b.repack([bad] * count)
    for _ in range(2):  # eager (after a repack), then as configured
        overwrite(b.fetch_raw(), b.lps)
        b.solve()
        r = b.fetch()
        assert (r.status == oracle.INFEASIBLE).all()
        assert (r.pivots == o["pivots"]).all() and (r.fallback == 0).all()
        assert (r.kkt_dual > 0).all() and (r.kkt_primal >= 0).all() and (r.kkt_primal <= 1e-9).all()
        for k in range(count):
            assert np.array_equal(r.basis[k], o["basis"])
    b.free()
    S.close()
