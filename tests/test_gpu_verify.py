"""GPU tests of the FP64 refinement check (kernel_verify.hip) against its CPU restatement
(tests/verify_ref.py) on the same final tableaux: the FP32 solves are bit-exact with the
oracle, so the oracle's FP32 tableau is the one the device checked.  Where the restatement
decides clearly (KKT measure 10x away from the tolerance), the device accepts / rejects the
same results, and an accepted result reports the restatement's FP64 objective and point.
"""
import numpy as np
import pytest

import oracle
import simplexprojects_amd as sa
from tests.common import load_netlib
from tests.test_verify_ref import STATUS, mixed_sense_lps
from tests.verify_ref import refine_check

pytestmark = pytest.mark.gpu
TOL = 1e-9


def compare(lps, r):
    decided = 0
    for k, lp in enumerate(lps):
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision="fp32", tab=True)
        assert r.pivots[k] == o["pivots"] or r.fallback[k], k
        if o["status"] not in STATUS:
            continue
        ref = refine_check(lp.A, lp.b, lp.c, lp.sense, STATUS[o["status"]], o["basis"],
                           o["tab"], o["nb"], o["unb_var"], float(np.abs(lp.A).max()), TOL)
        if ref["ok"] is None:
            assert r.fallback[k], k
            continue
        kk = max(ref["kkt_p"], ref.get("kkt_d", -1.0))
        if ref["ok"] and kk > 0.1 * TOL:
            continue
        if not ref["ok"] and STATUS[o["status"]] == "optimal" and kk < 10 * TOL:
            continue
        decided += 1
        assert bool(r.fallback[k]) == (not ref["ok"]), k
        if ref["ok"] and STATUS[o["status"]] == "optimal":
            assert abs(r.objective[k] - ref["objective"]) <= 1e-12 * (1 + abs(ref["objective"]))
            assert np.allclose(r.x[k], ref["x"], rtol=1e-12, atol=1e-12 * (1 + np.abs(ref["x"]).max()))
    return decided


def test_netlib_fp32_check_matches_restatement():
    nl = load_netlib()
    names = sorted(nl)
    lps = [sa.LP(nl[n][0], nl[n][1], nl[n][2]) for n in names]
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    assert compare(lps, r) >= 12
    # the singular FP32 bases are rejected and re-solved in FP64
    for name in ("BLEND", "SC50A", "SC105", "SC205"):
        assert r.fallback[names.index(name)], name
    S.close()


def test_mixed_sense_fp32_check_matches_restatement():
    lps = [sa.LP(A, b, c, s) for A, b, c, s in mixed_sense_lps(48, m=40, n=34, seed=5)]
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    assert compare(lps, r) >= 40
    S.close()


def test_generated_fp32_check_matches_restatement():
    lps = sa.gen_config(2, 2, 50, 48, 96, shape_idx=0, batch_count=1024)
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    assert compare(lps, r) >= 80
    S.close()


def test_large_lps_global_sweeps_match_restatement():
    # 205x203 LPs: their staged blocks (k ~ 110) exceed every tier's LDS, so the last tier
    # runs the sweeps from global memory (vectors in LDS, blocks read in place)
    lps = sa.gen_config(5, 5, 205, 203, 12, shape_idx=4, batch_count=1024)
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    assert compare(lps, r) >= 8
    S.close()


def test_two_phase_infeasible_certified_on_device():
    """FP32 INFEASIBLE results of the two-phase LPs (HiGHS: infeasible) are accepted by the
    device's Farkas check exactly where the restatement's certificate is clear, with the
    same violation and margin; a result the restatement cannot certify is re-solved."""
    from tests.common import load_highs
    g = load_highs(3)
    lps = []
    for grp in g["groups"]:
        lps += sa.gen_config(3, g["seed"], grp["m"], grp["n"], grp["count"],
                             shape_idx=grp["shape_idx"], first=grp["first"],
                             batch_count=grp["batch_count"])
    status = np.concatenate([np.asarray(grp["status"]) for grp in g["groups"]])
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    assert np.array_equal(r.status, status)
    decided = 0
    for k, lp in enumerate(lps):
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision="fp32", tab=True)
        assert o["status"] == oracle.INFEASIBLE
        ref = refine_check(lp.A, lp.b, lp.c, lp.sense, "infeasible", o["basis"], o["tab"],
                           o["nb"], -1, float(np.abs(lp.A).max()), TOL)
        clear_yes = ref["ok"] and ref["kkt_p"] < 0.1 * TOL and ref["kkt_d"] > 10 * np.sqrt(TOL)
        if clear_yes:
            decided += 1
            assert not r.fallback[k], k
            assert abs(r.kkt_dual[k] - ref["kkt_d"]) <= 1e-6 * ref["kkt_d"], k
            assert r.kkt_primal[k] <= 0.1 * TOL, k
        elif not ref["ok"]:
            assert r.fallback[k], k
    assert decided >= len(lps) // 2
    S.close()


def test_singular_final_basis_falls_back_from_before_its_last_pivot():
    # The 105x103 LPs of the mixed-size batch (seed 2).  LP 388's FP32 solve ends UNBOUNDED
    # on a basis that is singular in FP64 (cond ~5e7; its last pivot was on an element that
    # is tiny in exact arithmetic), so its basic solution does not refine and the FP64
    # fallback starts from the basis before that last pivot: the oracle's FP32 replay
    # stopped one pivot short.  The device result is the oracle's FP64 replay warm from that
    # basis, pivot for pivot, in under half the pivots of a cold re-solve.  LP 211's final
    # basis refines (only its ray fails), so it is re-solved warm from that basis.
    lps = sa.gen_config(2, 2, 105, 103, 1024, shape_idx=3, batch_count=1024)
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    S.close()
    fb = [k for k in range(len(lps)) if r.fallback[k]]
    assert 388 in fb and 211 in fb, fb
    for k, undo in ((388, True), (211, False)):
        lp = lps[k]
        o32 = oracle.solve(lp.A, lp.b, lp.c, precision="fp32")
        start = o32["basis"]
        if undo:
            start = oracle.solve(lp.A, lp.b, lp.c, precision="fp32",
                                 max_iter=o32["pivots"] - 1)["basis"]
        want = oracle.solve(lp.A, lp.b, lp.c, warm=start)
        assert r.status[k] == want["status"], k
        assert r.pivots[k] == want["pivots"], (k, r.pivots[k], want["pivots"])
        cold = oracle.solve(lp.A, lp.b, lp.c)
        assert r.status[k] == cold["status"], k
        if undo:
            assert r.pivots[k] < 0.5 * cold["pivots"], (r.pivots[k], cold["pivots"])


@pytest.mark.parametrize("config", [1, 2, 3])
@pytest.mark.parametrize("shape", [(6, 5), (40, 34), (105, 103), (205, 203)])
def test_tableaux_that_overflow_are_resolved(config, shape):
    """Rows scaled by 1e39 are infinite in FP32 and the pivots turn them into NaN: a basic
    solution that is not finite passes no check, and a reported optimum is finite.  (Not compared
    with the unscaled LP: the tolerances are relative to max |A|.)"""
    m, n = shape
    lps = []
    for k, lp in enumerate(sa.gen_config(config, 9, m, n, 8, shape_idx=1, batch_count=8)):
        scale = np.ones(m)
        scale[np.random.default_rng(k).permutation(m)[:1 + k * m // 8]] = 1e39
        lps.append(sa.LP(lp.A * scale[:, None], lp.b * scale, lp.c, lp.sense))
    S = sa.Solver(precision="fp32")
    r = S.solve(lps)
    S.close()
    for k, lp in enumerate(lps):
        o = oracle.solve(lp.A, lp.b, lp.c, lp.sense, precision="fp32", tab=True)
        # (an infeasible or unbounded one is certified by finite duals or a finite ray alone)
        if o["status"] == oracle.OPTIMAL and not np.isfinite(o["tab"][:, 0]).all():
            assert r.fallback[k], k
        if r.status[k] == sa.OPTIMAL:
            assert np.isfinite(r.objective[k]) and np.isfinite(r.x[k]).all(), k


def test_a_tableau_of_nan_is_no_optimum():
    # FP32: the first row is infinite, its pivot leaves NaN everywhere; the optimum is 5 at (1, 4)
    S = sa.Solver(precision="fp32")
    r = S.solve([sa.LP([[1e39, 1.0], [1.0, 1.0]], [1e39, 5.0], [1.0, 1.0])])
    S.close()
    assert (r.status[0], r.fallback[0], r.objective[0]) == (sa.OPTIMAL, 1, 5.0)
    assert r.x[0].tolist() == [1.0, 4.0]
