"""GPU tests of the instances chosen for the number of LPs of a bin: just below and above the
line, bit-equal results (each instance alone is compared with the oracle elsewhere), LPs that
only the route by size holds stay there, and batches routed for FP32 solve in FP64."""
import numpy as np
import pytest

import oracle
import simplexprojects_amd as sa

pytestmark = pytest.mark.gpu

CUS = 256  # MI355X

# precision, shape (m, n), LPs per CU at the line, route by size, instance beyond the line
RULES = [("fp64", (105, 103), 2, (3, 4), (3, 9)), ("fp64", (110, 110), 2, (3, 4), (3, 9)),
         ("fp64", (174, 142), 2, (3, 5), (3, 12)), ("fp64", (130, 90), 2, (3, 5), (3, 12)),
         ("fp32", (174, 142), 2, (4, 5), (3, 12)), ("fp32", (205, 203), 1, (4, 6), (3, 13)),
         ("fp32", (206, 206), 1, (4, 6), (3, 13))]


def batch(m, n, count, distinct=24):
    """count LPs, the last `distinct` of them different ones (the rest share one small LP's
    data: trivial, c <= 0)."""
    lps = sa.gen_config(2, 7, m, n, distinct, batch_count=distinct)
    A = np.ones((m, n))
    easy = sa.LP(A, np.ones(m), -np.ones(n))
    return [easy] * (count - distinct) + lps


def instances(info):
    return sorted((b["kernel"], b["param"], b["count"]) for b in info["bins"])


@pytest.mark.parametrize("precision,shape,per_cu,small,large", RULES)
def test_both_sides_of_the_line(precision, shape, per_cu, small, large):
    cus = CUS
    m, n = shape
    out = []
    for count, want in ((per_cu * cus, small), (per_cu * cus + 1, large)):
        lps = batch(m, n, count)
        S = sa.Solver(precision=precision, verify=precision == "fp32")
        b = S.upload(lps)
        assert instances(b.info()) == [(*want, count)]
        b.solve()
        out.append((b.fetch(), lps))
        b.free()
        S.close()
    (r0, l0), (r1, l1) = out
    for k in range(1, 25):
        for f in ("status", "pivots", "fallback", "objective"):
            assert getattr(r0, f)[-k] == getattr(r1, f)[-k], f
        assert np.array_equal(r0.x[-k], r1.x[-k]) and np.array_equal(r0.basis[-k], r1.basis[-k])
        if k <= 3 and not r1.fallback[-k]:
            o = oracle.solve(l1[-k].A, l1[-k].b, l1[-k].c, precision=precision)
            assert (r1.status[-k], r1.pivots[-k]) == (o["status"], o["pivots"])


def test_shapes_the_other_instance_does_not_hold():
    cus = CUS
    lps = batch(174, 142, 2 * cus + 1) + sa.gen_config(2, 7, 180, 140, 4, batch_count=4)
    S = sa.Solver(precision="fp64", verify=False)
    b = S.upload(lps)
    assert instances(b.info()) == [(3, 5, 4), (3, 12, 2 * cus + 1)]
    b.free()
    S.set(kernel="tile")  # a forced kernel keeps the route by size
    b = S.upload(lps)
    assert instances(b.info()) == [(3, 5, 2 * cus + 5)]
    b.free()
    S.close()


def test_warm_lists_keep_the_block_crash():
    cus = CUS
    lps = batch(105, 103, 2 * cus + 1)
    warm = sa.LP(lps[-1].A, lps[-1].b, lps[-1].c, warm_basis=np.arange(103, 103 + 105))
    S = sa.Solver(precision="fp64", verify=False)
    b = S.upload(lps[:-1] + [warm])
    assert instances(b.info()) == [(3, 4, 2 * cus + 1)]
    b.free()
    S.close()


@pytest.mark.parametrize("shape,count", [((27, 32), 8), ((105, 103), 8), ((174, 142), 8),
                                         ((205, 203), 300), ((250, 249), 2)])
def test_fp32_batch_solved_in_fp64(shape, count):
    lps = sa.gen_config(2, 3, *shape, min(count, 8), batch_count=8)
    lps = lps * (count // len(lps)) + lps[:count % len(lps)]
    S = sa.Solver(precision="fp32")
    b = S.upload(lps)
    S.set(precision="fp64")
    b.solve()
    r = b.fetch()
    T = sa.Solver(precision="fp64")
    want = T.solve(lps)
    for f in ("status", "pivots", "objective"):
        assert np.array_equal(getattr(r, f), getattr(want, f)), f
    for k in range(count):
        assert np.array_equal(r.x[k], want.x[k])
    b.free()
    S.close()
    T.close()


def test_lds_bins_stay_where_the_route_by_size_has_sixteen_bins():
    """With its other instance the batch would need a bin too many: it goes back to the route
    by size as it stands, LDS bins included."""
    lps = batch(174, 142, 2 * CUS + 1) + sa.gen_config(2, 7, 180, 140, 1, batch_count=1)
    for m in (230, 250, 270, 290, 310):
        for n in (10, 26, 42):
            lps += sa.gen_config(2, 7, m, n, 1, batch_count=1)
    S = sa.Solver(precision="fp64", verify=False)
    b = S.upload(lps)
    got = instances(b.info())
    assert len(got) == 16 and got[-1] == (3, 5, 2 * CUS + 2)
    assert all(kernel == 2 for kernel, _, _ in got[:-1]), got
    b.free()
    S.close()


@pytest.mark.parametrize("kernel", ["auto", "lds", "stream"])
def test_fp32_lds_batch_solved_in_fp64(kernel):
    """300x100 fits a CU's LDS in FP32 only."""
    lps = sa.gen_config(2, 3, 300, 100, 3, batch_count=3)
    S = sa.Solver(precision="fp32", kernel=kernel)
    b = S.upload(lps)
    assert b.info()["bins"][0]["kernel"] == (1 if kernel == "stream" else 2)
    S.set(precision="fp64")
    b.solve()
    r = b.fetch()
    T = sa.Solver(precision="fp64")
    want = T.solve(lps)
    for f in ("status", "pivots", "objective"):
        assert np.array_equal(getattr(r, f), getattr(want, f)), f
    b.free()
    S.close()
    T.close()
