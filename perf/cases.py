"""The workloads by which the solver's speed is judged, each through the entry points a
user's program calls.

A case names its LPs as "m x n : count" groups (`shapes`), the family they are drawn from
(`data`), the entry point (`api`) and the options.  Sizes are those of this repository's
benchmark configurations and tests (27x32, 50x48, 56x97, 74x83, 105x103, 174x142, 205x203,
and the random 3..250 sweep), plus one size beyond what the register file of a compute unit
holds.

  api "resident"  a batch uploaded once: one pass = Batch.solve() + Batch.fetch_raw()
  api "oneshot"   one pass = Solver.solve() on host LPs (upload, solve, download)
  api "shared"    one A and b, many objectives, all on the device: one pass =
                  blpg_solve_shared_A_noalloc on the current stream
  api "learned"   a resident batch of parametric-family LPs with a trained warm-start
                  network attached: one pass = inference + warm solve + results

Returned are all results a caller reads: status, objective, x, basis and the pivot counts.
(The check's residuals, kkt_primal and kkt_dual, are left out: they are the rounding noise
of the refinement itself, about 1e-16, and have no value to be compared with.)
"""
import ctypes
import math

import numpy as np
import torch

import simplexprojects_amd as sa


# ---------------------------------------------------------------------------------
# the cases

def listed():
    return [
        # one LP at a time, the latency a caller waits for: launches and the pivot chain
        {"name": "single_fp32", "api": "resident", "precision": "fp32", "verify": True,
         "data": "general", "shapes": "105x103:1"},
        # the smallest benchmark shape in FP64 without the check: the reference's own case
        {"name": "small_fp64", "api": "resident", "precision": "fp64", "verify": False,
         "data": "box", "shapes": "27x32:1024"},
        # the headline batch: four shapes, FP32 tableau with FP64 check and fallback
        {"name": "mixed_fp32", "api": "resident", "precision": "fp32", "verify": True,
         "data": "general", "shapes": "50x48:1024,56x97:1024,74x83:1024,105x103:1024"},
        # the same batch all in FP64, checked: what a user without FP32 runs
        {"name": "mixed_fp64", "api": "resident", "precision": "fp64", "verify": True,
         "data": "general", "shapes": "50x48:1024,56x97:1024,74x83:1024,105x103:1024"},
        # phase I + phase II with equality rows, infeasible and feasible LPs, FP32
        {"name": "twophase_fp32", "api": "resident", "precision": "fp32", "verify": True,
         "data": "twophase", "shapes": "174x142:1024,205x203:1024"},
        # the same in FP64, where 205x203 is the largest shape near the register file's size
        {"name": "twophase_fp64", "api": "resident", "precision": "fp64", "verify": True,
         "data": "twophase", "shapes": "174x142:512,205x203:512"},
        # odd and ragged sizes in one batch (many bins with few LPs each), FP32
        {"name": "ragged_fp32", "api": "resident", "precision": "fp32", "verify": True,
         "data": "general",
         "shapes": "3x5:64,17x9:64,33x61:96,47x130:48,65x64:96,91x37:64,113x127:48,"
                   "129x66:48,201x113:32,250x249:16"},
        # larger than registers or LDS hold: the tableau streams from HBM, few LPs, FP64
        {"name": "large_fp64", "api": "resident", "precision": "fp64", "verify": True,
         "data": "box", "shapes": "300x400:128"},
        # the reference's batch shape: one A and b, an objective per LP, device buffers
        {"name": "shared_fp64", "api": "shared", "precision": "fp64", "verify": False,
         "data": "family", "shapes": "74x83:4096"},
        # a parametric family re-solved from cold in FP32 (b and c move by 5%)
        {"name": "family_fp32", "api": "resident", "precision": "fp32", "verify": True,
         "data": "family", "shapes": "105x103:8192"},
        # the same kind of LPs with the learned warm start: inference, crash and repair
        {"name": "learned_fp32", "api": "learned", "precision": "fp32", "verify": True,
         "data": "family", "shapes": "105x103:4096"},
        # the blocking call on host LPs, as the reference's ComputeLP is called
        {"name": "oneshot_fp32", "api": "oneshot", "precision": "fp32", "verify": True,
         "data": "general", "shapes": "27x32:128,74x83:128"},
    ]


# LPs of one family share A; families per batch
_FAMILIES = 16
_COST_CAP = 5e10


def _groups(case):
    out = []
    for part in case["shapes"].split(","):
        mn, cnt = part.split(":")
        m, n = mn.split("x")
        out.append((int(m), int(n), int(cnt)))
    return out


# pivots an LP takes, as a multiple of min(m, n): measured means of the families below
_PIVOTS = {"box": 0.35, "family": 0.3, "general": 1.4, "twophase": 2.2}


def _flops(case):
    f = _PIVOTS[case["data"]]
    return sum(cnt * max(1.0, f * min(m, n)) * 2.0 * (m + 1) * (n + 1)
               for m, n, cnt in _groups(case))


def draw(rng):
    """A case of the listed ranges: 1 to 5 shapes of 3..250 rows and columns (one shape up
    to 400 for "box" in FP64), 1 to 8192 LPs, every api, precision and data family."""
    def logint(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    api = rng.choice(["resident", "resident", "resident", "resident", "shared", "learned", "oneshot"])
    precision, verify = rng.choice([("fp32", True), ("fp32", True), ("fp64", True), ("fp64", False)])
    data = rng.choice(["box", "general", "general", "twophase", "family"])
    groups = rng.choice([1, 1, 2, 3, 5])
    lo, hi, most = 3, 250, 2048
    if api == "shared":
        precision, verify, data, groups, hi, most = "fp64", False, "family", 1, 110, 8192
    elif api == "learned":
        precision, verify, data, groups, lo, hi, most = "fp32", True, "family", 1, 16, 120, 4096
    elif api == "oneshot":
        most = 256
    elif data == "box" and precision == "fp64" and rng.random() < 0.5:
        groups, hi, most = 1, 400, 256
    if data == "twophase":
        lo = 8
    shapes = []
    for _ in range(groups):
        m = logint(lo, hi)
        n = logint(max(lo, m // 3), min(hi, 3 * m))
        cnt = logint(1, most)
        if api == "learned":
            cnt = max(_FAMILIES, cnt)
        if api == "shared":
            cnt = min(cnt, 30000000 // (8 * (m + 3 * n + 64)) // 2)
        # host arrays of a drawn case stay below the largest listed case's
        cnt = max(1 if api != "learned" else _FAMILIES, min(cnt, int(3e7 / (m * n)) // groups))
        shapes.append([m, n, cnt])
    case = {"api": api, "precision": precision, "verify": verify, "data": data}
    while True:
        case["shapes"] = ",".join("%dx%d:%d" % tuple(s) for s in shapes)
        w = 4.0 if precision == "fp64" else 1.0
        if _flops(case) * w <= _COST_CAP / 2 or all(s[2] <= 1 for s in shapes):
            return case
        for s in shapes:
            s[2] = max(1, s[2] // 2)


# ---------------------------------------------------------------------------------
# the LPs: maximise c x, A x (<=, =, >=) b, x >= 0

def _lps(case, seed):
    """Per group: (A, b, c, sense or None, family ids or None); A is (count, m, n), or
    (families, m, n) for the parametric families."""
    rng = np.random.default_rng([seed, 1])
    out = []
    for m, n, k in _groups(case):
        data = case["data"]
        if data == "box":  # A >= 0: bounded, a few pivots
            A = np.where(rng.random((k, m, n)) < 0.3, 0.0, rng.random((k, m, n)))
            A[:, 0, :] += 0.05  # no empty column
            out.append((A, 1 + 9 * rng.random((k, m)), rng.random((k, n)), None, None))
        elif data == "general":  # signed A, 10% of b zero (degenerate), many LPs unbounded
            A = np.where(rng.random((k, m, n)) < 0.4, 0.0, 2 * rng.random((k, m, n)) - 1)
            b = 10 * rng.random((k, m))
            b[np.argsort(rng.random((k, m)), axis=1) < m // 10] = 0.0
            c = rng.standard_normal((k, n))
            for i in range(0, k, 20):  # 5% planted unbounded
                j = int(rng.integers(n))
                A[i, :, j] = -np.abs(A[i, :, j])
                c[i, j] = abs(c[i, j]) + 0.1
            out.append((A, b, c, None, None))
        elif data == "twophase":  # 30% '=' rows; even LPs feasible and bounded, odd random
            A = np.where(rng.random((k, m, n)) < 0.5, 0.0, 2 * rng.random((k, m, n)) - 1)
            b = 5 * rng.standard_normal((k, m))
            sense = np.zeros((k, m), np.int8)
            rank = np.argsort(np.argsort(rng.random((k, m - 1)), axis=1), axis=1)
            # fewer '=' rows than columns, or a random system has no solution at all
            neq = min(int(round(0.3 * m)), n // 2)
            sense[:, :m - 1][rank < neq] = 1
            feas = np.arange(k) % 2 == 0
            ge = (rank >= neq) & (rank < neq + (m - 1 - neq) // 2) & feas[:, None]
            sense[:, :m - 1][ge] = 2
            x = 2 * rng.random((k, n))
            slack = 0.1 + 0.9 * rng.random((k, m))
            A[feas, -1] = 1.0
            bf = np.matmul(A[feas], x[feas][:, :, None])[:, :, 0]
            bf += np.where(sense[feas] == 0, slack[feas], np.where(sense[feas] == 2, -slack[feas], 0.0))
            bf[:, -1] = x[feas].sum(1) + 5.0
            b[feas] = bf
            out.append((A, b, rng.standard_normal((k, n)), sense, None))
        else:  # parametric families: A fixed per family, b and c scaled by 1 + 0.05 N(0,1)
            nf = 1 if case["api"] == "shared" else min(_FAMILIES, k)
            A = np.where(rng.random((nf, m, n)) < 0.3, 0.0, rng.random((nf, m, n)))
            A[:, 0, :] += 0.05
            fam = (np.arange(k) * nf // k).astype(np.int64)
            b0, c0 = 1 + 9 * rng.random((nf, m)), rng.random((nf, n))
            if case["api"] == "shared":  # one b, an objective per LP
                b = np.broadcast_to(b0[0], (k, m))
                c = rng.random((k, n))
            else:
                b = b0[fam] * (1 + 0.05 * rng.standard_normal((k, m)))
                c = c0[fam] * (1 + 0.05 * rng.standard_normal((k, n)))
            out.append((A, b, c, None, fam))
    return out


def _objects(groups):
    lps = []
    for A, b, c, sense, fam in groups:
        for i in range(len(c)):
            lps.append(sa.LP(A[i] if fam is None else A[fam[i]], b[i], c[i],
                             None if sense is None else sense[i],
                             family=-1 if fam is None else int(fam[i])))
    return lps


# ---------------------------------------------------------------------------------

def prepare(case, seed):
    groups = _lps(case, seed)
    if case["api"] == "shared":
        A, b, c, _, _ = groups[0]
        m, n = A.shape[1:]
        dev = lambda v: torch.tensor(np.ascontiguousarray(v), dtype=torch.float64, device="cuda")
        k = len(c)
        f64 = lambda *s: torch.empty(s, dtype=torch.float64, device="cuda")
        i32 = lambda *s: torch.empty(s, dtype=torch.int32, device="cuda")
        return {"api": "shared", "lib": sa.load_library(), "m": m, "n": n, "k": k,
                "A": dev(A[0]), "b": dev(b[0]), "C": dev(c), "status": i32(k),
                "objective": f64(k), "x": f64(k, n), "basis": i32(k, m), "pivots": i32(k)}
    lps = _objects(groups)
    solver = sa.Solver(precision=case["precision"], verify=case["verify"])
    state = {"api": case["api"], "solver": solver}
    if case["api"] == "oneshot":
        state["lps"] = lps
        return state
    if case["api"] == "learned":
        # the network is trained on other instances of the same families, on cold FP64 bases
        m, n, k = _groups(case)[0]
        A, b, c, _, fam = groups[0]
        nf = len(A)
        rng = np.random.default_rng([seed, 2])
        pick = rng.integers(0, k, 64 * nf)
        train = [sa.LP(A[fam[i]], b[i] * (1 + 0.02 * rng.standard_normal(m)),
                       c[i] * (1 + 0.02 * rng.standard_normal(n)), None, family=int(fam[i]))
                 for i in pick]
        train.sort(key=lambda lp: lp.family)
        label = sa.Solver(precision="fp64", verify=False)
        bases = label.solve(train).basis
        label.close()
        state["model"] = sa.WarmStart(solver, nf, m, n, seed=4, steps=100, lr=3e-3,
                                      weight_decay=1e-2)
        state["model"].train(train, bases)
    state["batch"] = solver.upload(lps)
    state["nx"], state["nb"] = sum(lp.n for lp in lps), sum(lp.m for lp in lps)
    if case["api"] == "learned":
        state["batch"].set_warmstart(state["model"])
    return state


class _Pinned:
    """An array view of a batch's pinned results that keeps the batch alive."""

    def __init__(self, batch, ptr, n, typestr):
        self.batch = batch
        self.__array_interface__ = {"data": (ctypes.cast(ptr, ctypes.c_void_p).value, True),
                                    "shape": (n,), "typestr": typestr, "version": 3}


def run(state):
    if state["api"] == "shared":
        s = state
        rc = s["lib"].blpg_solve_shared_A_noalloc(
            s["m"], s["n"], s["A"].data_ptr(), s["b"].data_ptr(), None, s["C"].data_ptr(),
            s["k"], s["status"].data_ptr(), s["objective"].data_ptr(), s["x"].data_ptr(),
            s["basis"].data_ptr(), s["pivots"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise sa.BlpgError(rc, s["lib"].blpg_last_error(None).decode())
        return {k: s[k] for k in ("status", "objective", "x", "basis", "pivots")}
    if state["api"] == "oneshot":
        r = state["solver"].solve(state["lps"])
        return {"status": r.status, "pivots": r.pivots, "phase1_pivots": r.phase1_pivots,
                "fallback": r.fallback, "objective": r.objective, "x": np.concatenate(r.x),
                "basis": np.concatenate(r.basis)}
    batch = state["batch"]
    batch.solve()
    r = batch.fetch_raw()  # waits; the results are in the batch's pinned host buffers
    k = r.count
    i32 = lambda p, n: np.asarray(_Pinned(batch, p, n, "<i4"))
    f64 = lambda p, n: np.asarray(_Pinned(batch, p, n, "<f8"))
    return {"status": i32(r.status, k), "pivots": i32(r.pivots, k),
            "phase1_pivots": i32(r.phase1_pivots, k), "fallback": i32(r.fallback_used, k),
            "objective": f64(r.objective, k), "x": f64(r.x, state["nx"]),
            "basis": i32(r.basis, state["nb"])}


def work(case):
    """Inputs read once, results written once; two flops per entry of the condensed tableau
    and pivot (the mean pivot counts of the data families)."""
    total = 0
    for m, n, k in _groups(case):
        na = min(_FAMILIES, k) if case["data"] == "family" else k
        if case["api"] == "shared":
            na = 1
        total += 8 * na * m * n + k * (8 * (m + n) + 8 * n + 4 * m + 24)
    return {"bytes": float(total), "flops": float(_flops(case))}


# ---------------------------------------------------------------------------------
# 64-bit results without the framework's code: the textbook primal simplex method
# (Dantzig's rule, as the solver's contract states it) on whole batches in torch, then the
# final basis solved against the input data

def _simplex64(A, b, c):
    """(x, objective, basis, all optimal?) of maximise c x, A x <= b, x >= 0 with b >= 0,
    per LP of the batch; None when an LP degenerates so long that the solver would change its
    pivot rule, or does not end."""
    k, m, n = A.shape
    dev = A.device
    T = torch.zeros(k, m + 1, n + 1, dtype=torch.float64, device=dev)
    T[:, 0, 1:] = -c
    T[:, 1:, 0] = b
    T[:, 1:, 1:] = A
    bs = (n + torch.arange(m, device=dev)).repeat(k, 1)
    nb = torch.arange(n, device=dev).repeat(k, 1)
    live = torch.arange(k, device=dev)
    deg = torch.zeros(k, dtype=torch.int64, device=dev)
    final = [None, None, torch.zeros(k, dtype=torch.bool, device=dev)]
    end_bs = bs.clone()
    end_obj = torch.zeros(k, dtype=torch.float64, device=dev)
    for _ in range(50 * (m + n) + 1000):
        d, s = T[:, 0, 1:].min(dim=1)
        opt = ~(d < -1e-9)
        col = torch.gather(T, 2, (s + 1)[:, None, None].expand(-1, m + 1, 1))[:, :, 0]
        a = col[:, 1:]
        beta = T[:, 1:, 0].clamp(min=0.0)
        th = beta / torch.where(a > 1e-9, a, torch.ones_like(a))
        key = torch.where(th > 0, th, -a)
        key = torch.where(a > 1e-9, key, torch.full_like(key, math.inf))
        kv, r = key.min(dim=1)
        unb = ~opt & torch.isinf(kv)
        done = opt | unb
        if bool(done.any()):
            w = live[done]
            end_bs[w] = bs[done]
            end_obj[w] = T[done, 0, 0]
            final[2][w] = opt[done]
            keep = ~done
            if not bool(keep.any()):
                break
            T, bs, nb, live, deg = T[keep], bs[keep], nb[keep], live[keep], deg[keep]
            col, r, s, kv = col[keep], r[keep], s[keep], kv[keep]
        deg = torch.where(kv > 0, torch.zeros_like(deg), deg + 1)
        if int(deg.max()) >= 50:
            return None
        q = torch.arange(len(live), device=dev)
        rp = 1.0 / col[q, r + 1]
        prow = T[q, r + 1] * rp[:, None]
        prow[q, s + 1] = rp
        T[q, :, s + 1] = 0.0
        T = torch.baddbmm(T, -col[:, :, None], prow[:, None, :])
        T[q, r + 1] = prow
        e, lv = nb[q, s].clone(), bs[q, r].clone()
        bs[q, r], nb[q, s] = e, lv
    else:
        return None
    # basic solution of the final basis from the data: columns of [A I]
    full = torch.cat([A, torch.eye(m, dtype=torch.float64, device=dev).expand(k, m, m)], dim=2)
    B = torch.gather(full, 2, end_bs[:, None, :].expand(-1, m, -1))
    xb = torch.linalg.solve(B, b[:, :, None])[:, :, 0]
    x = torch.zeros(k, n + m, dtype=torch.float64, device=dev)
    x.scatter_(1, end_bs, xb)
    x = x[:, :n]
    return x, (c * x).sum(1), end_obj, final[2]


def exact(case, seed):
    """objective and x.  None for two-phase LPs (an infeasible one has no x) and for FP32
    batches with an unbounded LP, whose last vertex depends on the FP32 path."""
    if case["data"] == "twophase":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    up = lambda v: torch.tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)
    xs, objs = [], []
    for A, b, c, _, fam in _lps(case, seed):
        A = up(A)
        if fam is not None:
            A = A[torch.from_numpy(fam).to(dev)]
        got = _simplex64(A, up(b), up(c))
        if got is None:
            return None
        x, obj, _, opt = got
        if case["precision"] == "fp32" and not bool(opt.all()):
            return None
        xs.append(x.reshape(-1))
        objs.append(obj)
    x, obj = torch.cat(xs).cpu().numpy(), torch.cat(objs).cpu().numpy()
    if case["api"] == "shared":
        x = x.reshape(len(obj), -1)
    return {"objective": obj, "x": x}
