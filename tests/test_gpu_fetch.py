"""GPU tests of a fetch's host copy: the first fetch of a batch copies the results, later
solves have the check kernels write them; both must hold the same bytes, for every way an
LP can end (each check tier, verified, failed and re-solved, infeasible, unbounded,
iteration limit), and a solve without a check must not leave an older solve's results."""
import numpy as np
import pytest

import simplexprojects_amd as sa
from tests.test_gpu_check_fit import overwrite

pytestmark = pytest.mark.gpu


def lps_of(kind):
    rng = np.random.default_rng(5)
    if kind == "one":
        return sa.gen_config(2, 2, 105, 103, 1, shape_idx=3, batch_count=1024)
    if kind == "bins":
        out = []
        for si, (m, n) in enumerate([(50, 48), (56, 97), (74, 83), (105, 103)]):
            out += sa.gen_config(2, 2, m, n, 300, shape_idx=si, batch_count=1024)
        return out
    if kind == "twophase":
        return sa.gen_config(3, 3, 205, 203, 40, shape_idx=1, batch_count=8192)
    out = []  # unbounded, infeasible, one row, one column, degenerate
    for m, n in [(1, 1), (1, 7), (9, 1), (17, 30), (64, 65)]:
        A = rng.integers(0, 5, (m, n)) + 1.0
        c = rng.integers(1, 9, n) * 1.0
        out.append(sa.LP(A, np.ones(m), c))
        out.append(sa.LP(-A, np.ones(m), c))
        out.append(sa.LP(A, -np.ones(m), c))
        out.append(sa.LP(A, np.zeros(m), c))
    return out


def same(a, b):
    for f in ("status", "pivots", "phase1_pivots", "fallback", "objective", "kkt_primal",
              "kkt_dual"):
        assert np.array_equal(getattr(a, f), getattr(b, f), equal_nan=True), f
    for k in range(len(a)):
        assert np.array_equal(a.x[k], b.x[k]) and np.array_equal(a.basis[k], b.basis[k])


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("kind", ["one", "bins", "twophase", "ends"])
def test_written_equals_copied(kind, precision, graph):
    S = sa.Solver(precision=precision, verify=True, use_graph=graph)
    b = S.upload(lps_of(kind))
    b.solve()
    ref = b.fetch()  # copied
    for _ in range(3):
        b.solve()
        same(b.fetch(), ref)  # written by the check
    same(b.fetch(), ref)  # once more, without a solve
    b.free()
    S.close()


def test_options_between_solves():
    """Iteration limits and no check after a checked solve: each fetch is its own solve's."""
    lps = lps_of("bins")[:400]
    S = sa.Solver(precision="fp64", verify=True)
    b = S.upload(lps)
    b.solve()
    ref = b.fetch()
    for verify, iters in [(True, 3), (False, 3), (True, 0), (False, 0), (True, 0)]:
        S.set(verify=int(verify), max_iter=iters)
        T = sa.Solver(precision="fp64", verify=verify, max_iter=iters)
        t = T.upload(lps)
        t.solve()
        want = t.fetch()
        b.solve()
        same(b.fetch(), want)
        t.free()
        T.close()
    same(b.fetch(), ref)
    b.free()
    S.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("kind", ["one", "bins", "twophase", "ends", "limit", "narrow"])
def test_later_solves_write_every_result(kind, precision, graph):
    """The host copy holds other values before each later solve: every result of every LP is
    the solve's own.  limit: iteration limits (FP32: all re-solved); narrow: bins of LPs with
    fewer columns than rows, whose check has fewer tiers."""
    if kind == "narrow":
        batches = [[lp] * 3 for lp in lps_of("ends") if lp.n == 1]
        batches += [sa.gen_config(2, 4, m, n, 3, batch_count=3) for m, n in [(5, 3), (60, 35), (78, 75)]]
    else:
        batches = [lps_of("bins" if kind == "limit" else kind)]
    S = sa.Solver(precision=precision, verify=True, use_graph=graph, max_iter=3 if kind == "limit" else 0)
    for lps in batches:
        b = S.upload(lps)
        b.solve()
        ref = b.fetch()  # copied
        for _ in range(2):
            overwrite(b.fetch_raw(), lps)
            b.solve()
            same(b.fetch(), ref)
        b.free()
    S.close()


def test_a_fetch_leaves_the_solves_results_as_they_are():
    """Options set after a solve, and what a caller writes into the fetched arrays, do not
    reach the next fetch of the same solve, whether the check wrote them or a copy did."""
    S = sa.Solver(precision="fp64", verify=True)
    b = S.upload(lps_of("bins")[:40])
    b.solve()
    ref = b.fetch()
    for _ in range(2):  # copied, written by the check
        S.set(verify=0)
        r = b.fetch()
        assert (r.kkt_primal == -1).all() and (r.kkt_dual == -1).all()
        S.set(verify=1)
        same(b.fetch(), ref)
        raw = b.fetch_raw()
        for f in ("status", "pivots", "phase1_pivots", "fallback_used", "objective"):
            np.ctypeslib.as_array(getattr(raw, f), shape=(40,))[:] = -77
        same(b.fetch(), ref)
        b.solve()
    b.free()
    S.close()


@pytest.mark.parametrize("graph", [False, True])
def test_options_after_an_unchecked_solve(graph):
    """Whether the results are checked ones, and of which precision, is a matter of the solve:
    after an unchecked one a fetch reports no older solve's objective or residuals."""
    lps = lps_of("bins")[:40]
    S = sa.Solver(precision="fp64", verify=True, use_graph=graph)
    b = S.upload(lps)
    b.solve()
    b.fetch()
    S.set(verify=0, max_iter=3)
    T = sa.Solver(precision="fp64", verify=False, max_iter=3)
    t = T.upload(lps)
    t.solve()
    want = t.fetch()
    b.solve()
    S.set(verify=1)
    same(b.fetch(), want)
    assert b.info()["verify_ms"] <= 0
    t.free()
    b.free()
    S.close()
    T.close()


def test_precisions_in_turn_around_a_repack():
    """An FP32 graph replayed after a repacked batch was solved in FP64 without a check: FP32
    results are checked ones whatever ran in between."""
    lps = lps_of("bins")[:40]
    S = sa.Solver(precision="fp32", verify=False, use_graph=True)
    b = S.upload(lps)
    b.solve()
    ref = b.fetch()
    b.solve()  # captured again, writing the host copy
    T = sa.Solver(precision="fp64", verify=False)
    t = T.upload(lps)
    t.solve()
    want = t.fetch()
    S.set(precision="fp64")
    b.repack(lps)
    b.solve()
    same(b.fetch(), want)
    S.set(precision="fp32")
    b.solve()
    same(b.fetch(), ref)
    t.free()
    b.free()
    S.close()
    T.close()
