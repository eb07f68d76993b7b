"""The work that programs have this library do, as timed cases.

Every case goes through the public Python entry points (Solver, Batch, dspike_core_host, host_solve):

  step      factor a matrix that is in device memory and solve for its right-hand sides (one new
            matrix per step, as in a time-stepping or Newton loop); the solver object is kept, so a
            repeated step replays its captured solve
  resident  solve for right-hand sides with factors that are already in device memory
  batch     factor and solve many independent systems of uneven size in one call
  host      the reference's top-level entry point: host arrays in, host solution out
  band      the reference's reduced-system solver slot: banded LU with partial pivoting, host arrays

Matrices are random banded CSR, as the benchmark's: each in-band off-diagonal entry present with
probability `fill`, values U[-1, 1], diagonal max(dom * sum|off-diagonal| + add, 1); right-hand
sides U[-1, 1].  Solves end at a per-column relative residual of `tol`.
"""
import math

import numpy as np
import torch

import hspike_amd as hs

DEV = "cuda:0"
BATCH_K = (4, 8, 16, 32, 64)


def listed():
    return [
        # a small pentadiagonal system on the reference's four partitions: chain latency and launches
        dict(name="penta_fp64_small", kind="step", prec="fp64", cplx=False, n=10_000, kl=2, ku=2, fill=1.0, dom_lo=1.0,
             dom_hi=1.0, add=1.0, nrhs=1, parts=4, tol=1e-10),
        # repeated right-hand sides on a small resident matrix: the shortest call
        dict(name="resident_small", kind="resident", prec="mixed", cplx=False, n=20_000, kl=32, ku=32, fill=0.3,
             dom_lo=1.05, dom_hi=1.05, add=0.0, nrhs=4, parts=0, tol=1e-10),
        # a large resident matrix, unequal bandwidths, odd sizes, right-hand sides past two column tiles
        dict(name="resident_asym_fp64", kind="resident", prec="fp64", cplx=False, n=400_009, kl=50, ku=23, fill=0.25,
             dom_lo=1.1, dom_hi=1.1, add=0.0, nrhs=33, parts=0, tol=1e-10),
        # one million rows, half-bandwidth 64, 16 right-hand sides, in both precisions
        dict(name="step_1m_mixed", kind="step", prec="mixed", cplx=False, n=1_000_000, kl=64, ku=64, fill=0.15,
             dom_lo=1.05, dom_hi=1.05, add=0.0, nrhs=16, parts=0, tol=1e-10),
        dict(name="step_1m_fp64", kind="step", prec="fp64", cplx=False, n=1_000_000, kl=64, ku=64, fill=0.15,
             dom_lo=1.05, dom_hi=1.05, add=0.0, nrhs=16, parts=0, tol=1e-10),
        # two million rows, half-bandwidth 128, 64 right-hand sides refined to 1e-12: the largest system
        dict(name="step_2m_mixed", kind="step", prec="mixed", cplx=False, n=2_000_000, kl=128, ku=128, fill=0.2,
             dom_lo=1.01, dom_hi=2.0, add=0.0, nrhs=64, parts=0, tol=1e-12),
        # complex128 values, odd sizes
        dict(name="step_complex", kind="step", prec="mixed", cplx=True, n=200_003, kl=40, ku=40, fill=0.3, dom_lo=1.2,
             dom_hi=1.2, add=0.0, nrhs=7, parts=0, tol=1e-10),
        # the widest bands (half-bandwidth above 128)
        dict(name="step_wide", kind="step", prec="mixed", cplx=False, n=60_001, kl=200, ku=200, fill=0.3, dom_lo=1.2,
             dom_hi=1.2, add=0.0, nrhs=16, parts=0, tol=1e-10),
        # an eighth of the benchmark's batch: 512 systems of 1e3 to 2e5 rows
        dict(name="batch_512_mixed", kind="batch", prec="mixed", nsys=512, n_lo=1_000, n_hi=200_000, fill=0.3, dom=1.1,
             nrhs_hi=8, tune="throughput", draw=20261204, tol=1e-10),
        # a batch of few, smaller systems in FP64, tuned for latency
        dict(name="batch_48_fp64", kind="batch", prec="fp64", nsys=48, n_lo=1_000, n_hi=40_000, fill=0.3, dom=1.1,
             nrhs_hi=8, tune="latency", draw=9, tol=1e-10),
        # the reference's entry point on a heptadiagonal matrix and two right-hand sides
        dict(name="host_hepta", kind="host", n=100_000, kl=3, ku=3, fill=1.0, dom=1.1, nrhs=2, tol=1e-10),
        # the reduced system of 32 partitions at half-bandwidth 64
        dict(name="band_reduced", kind="band", parts=32, k=64, nrhs=16, tol=1e-10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "resident", "resident", "batch", "batch", "host", "band"])
    if kind == "batch":
        return dict(kind=kind, prec=rng.choice(["mixed", "fp64"]), nsys=_log(rng, 16, 256), n_lo=1_000,
                    n_hi=_log(rng, 20_000, 120_000), fill=round(rng.uniform(0.15, 0.5), 3), dom=1.1, nrhs_hi=rng.randint(1, 8),
                    tune=rng.choice(["throughput", "latency"]), draw=rng.randrange(1 << 30), tol=1e-10)
    if kind == "host":
        return dict(kind=kind, n=_log(rng, 10_000, 200_000), kl=rng.randint(1, 16), ku=rng.randint(1, 16), fill=1.0, dom=1.1,
                    nrhs=rng.randint(1, 8), tol=1e-10)
    if kind == "band":
        return dict(kind=kind, parts=rng.randint(4, 32), k=rng.randint(3, 64), nrhs=rng.randint(1, 16), tol=1e-10)
    cplx = rng.random() < 0.2
    prec = rng.choice(["mixed", "mixed", "fp64"])
    kl = _log(rng, 2, 256)
    ku = kl if rng.random() < 0.5 else max(1, min(256, int(kl * rng.uniform(0.5, 1.5))))
    k = max(kl, ku)
    n_hi = 60_000 if k > 128 else (300_000 if cplx else 800_000)
    if cplx and k > 64:
        n_hi = 30_000
    return dict(kind=kind, prec=prec, cplx=cplx, n=_log(rng, 10_000, n_hi), kl=kl, ku=ku, fill=round(rng.uniform(0.15, 0.5), 3),
                dom_lo=1.1, dom_hi=round(rng.uniform(1.1, 2.0), 2), add=0.0, nrhs=_log(rng, 1, 32 if cplx else 64), parts=0,
                tol=1e-10)


# ------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, cplx, *shape):
    v = torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64).mul_(2.0).sub_(1.0)
    if not cplx:
        return v
    return torch.complex(v, torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64).mul_(2.0).sub_(1.0))


def _bands(g, sizes, kl, ku, fill, dom_lo, dom_hi, add, cplx):
    """Diagonals of the matrices of `sizes` rows, stacked: values [rows, kl + 1 + ku] (zero where there
    is no entry), mask of the entries, first row of each matrix."""
    rows, width = sum(sizes), kl + 1 + ku
    ends = torch.tensor(np.cumsum(sizes), device=DEV)
    at = torch.arange(rows, device=DEV)
    last = ends[torch.searchsorted(ends, at, right=True)]
    size = torch.tensor(sizes, device=DEV)[torch.searchsorted(ends, at, right=True)]
    own = at - (last - size)                                           # row inside its matrix
    col = own[:, None] + torch.arange(-kl, ku + 1, device=DEV)
    mask = (col >= 0) & (col < size[:, None])
    if fill < 1.0:
        mask &= torch.rand(rows, width, generator=g, device=DEV) < fill
    mask[:, kl] = False
    val = _uniform(g, cplx, rows, width).mul_(mask)
    dom = torch.rand(rows, generator=g, device=DEV, dtype=torch.float64) * (dom_hi - dom_lo) + dom_lo
    val[:, kl] = (dom * val.abs().sum(1) + add).clamp_min(1.0).to(val.dtype)
    mask[:, kl] = True
    return val, mask, col


def _csr(val, mask, col):
    rowptr = torch.zeros(val.shape[0] + 1, dtype=torch.int32, device=DEV)
    rowptr[1:] = mask.sum(1).cumsum(0)
    return rowptr, col[mask].to(torch.int32), val[mask]


def _single(case, seed):
    """Diagonals of a step / resident / host case and its right-hand sides (nrhs x n)."""
    g = _gen(seed)
    cplx = case.get("cplx", False)
    lo, hi = (case["dom"], case["dom"]) if "dom" in case else (case["dom_lo"], case["dom_hi"])
    val, mask, col = _bands(g, [case["n"]], case["kl"], case["ku"], case["fill"], lo, hi, case.get("add", 0.0), cplx)
    return val, mask, col, _uniform(g, cplx, case["nrhs"], case["n"])


def _sizes(case):
    """(n, half-bandwidth, right-hand sides) of a batch's systems."""
    r = np.random.RandomState(case["draw"])
    n = np.exp(r.uniform(np.log(case["n_lo"]), np.log(case["n_hi"]), case["nsys"])).astype(np.int64)
    k = r.choice(np.array(BATCH_K), case["nsys"])
    m = r.randint(1, case["nrhs_hi"] + 1, case["nsys"])
    return [(int(a), int(b), int(c)) for a, b, c in zip(n, k, m)]


def _batch(case, seed):
    """Per half-bandwidth: its systems' indices, their stacked diagonals; and the right-hand sides of
    all systems in one array, system after system."""
    g = _gen(seed)
    spec = _sizes(case)
    groups = []
    for k in BATCH_K:
        ids = [i for i, s in enumerate(spec) if s[1] == k]
        if ids:
            groups.append((k, ids, _bands(g, [spec[i][0] for i in ids], k, k, case["fill"], case["dom"], case["dom"], 0.0, False)))
    return spec, groups, _uniform(g, False, sum(n * m for n, _, m in spec))


def _reduced(case, seed):
    """A reduced system of `parts` partitions and half-bandwidth k, dense: unit diagonal, per partition the
    columns W of its left neighbour's bottom tip and V of its right neighbour's top tip, decaying with the
    distance from the tip; near tips strong enough that rows are interchanged now and then."""
    r = np.random.RandomState(seed % (1 << 32))
    P, k = case["parts"], case["k"]
    n = 2 * k * P
    R = np.zeros((n, n))
    d = np.abs(np.arange(k)[:, None] - np.arange(k)[::-1][None, :])
    for p in range(P):
        top, bot = slice(2 * k * p, 2 * k * p + k), slice(2 * k * p + k, 2 * k * p + 2 * k)
        if p > 0:
            c = slice(2 * k * p - k, 2 * k * p)
            R[top, c] = 0.3 * r.uniform(-1, 1, (k, k)) * np.exp(-d.T / 8.0)
            R[bot, c] = 1e-6 * r.uniform(-1, 1, (k, k))
        if p + 1 < P:
            c = slice(2 * k * (p + 1), 2 * k * (p + 1) + k)
            R[bot, c] = 0.3 * r.uniform(-1, 1, (k, k)) * np.exp(-d / 8.0)
            R[top, c] = 1e-6 * r.uniform(-1, 1, (k, k))
    np.fill_diagonal(R, 1.0)
    return R, r.uniform(-1, 1, (n, case["nrhs"]))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "band":
        R, B = _reduced(case, seed)
        at, col = np.nonzero(R)
        rowptr = np.zeros(R.shape[0] + 1, np.int32)
        np.add.at(rowptr, at + 1, 1)
        return dict(kind=kind, A=hs.CSRMatrix(R.shape[0], np.cumsum(rowptr), col, R[at, col]), B=np.asfortranarray(B))
    if kind == "host":
        val, mask, col, B = _single(case, seed)
        rowptr, colind, aij = (t.cpu().numpy() for t in _csr(val, mask, col))
        return dict(kind=kind, A=hs.CSRMatrix(case["n"], rowptr, colind, aij), B=np.asfortranarray(B.cpu().numpy().T))
    if kind == "batch":
        spec, groups, B = _batch(case, seed)
        X = torch.zeros_like(B)
        first = np.concatenate([[0], np.cumsum([n * m for n, _, m in spec])])
        systems = [None] * len(spec)
        for k, ids, (val, mask, col) in groups:
            rowptr, colind, aij = _csr(val, mask, col)
            r0 = np.concatenate([[0], np.cumsum([spec[i][0] for i in ids])])
            e0 = rowptr[torch.from_numpy(r0).to(DEV)].tolist()
            for q, i in enumerate(ids):
                n, _, m = spec[i]
                s = slice(int(first[i]), int(first[i + 1]))
                systems[i] = dict(n=n, nrhs=m, rowptr=rowptr[r0[q]:r0[q + 1] + 1] - e0[q], colind=colind[e0[q]:e0[q + 1]].clone(),
                                  aij=aij[e0[q]:e0[q + 1]].clone(), b=B[s].view(m, n), x=X[s].view(m, n))
        bt = hs.Batch(case["prec"], tol=case["tol"], graph=True, tune=case["tune"])
        torch.cuda.synchronize()
        return dict(kind=kind, batch=bt, prep=bt.prepare(systems), X=X)
    val, mask, col, B = _single(case, seed)
    csr = _csr(val, mask, col)
    del val, mask, col
    torch.cuda.synchronize()
    s = hs.Solver(case["prec"], partitions=case["parts"], tol=case["tol"], graph=True)
    s.set_matrix_dev(case["n"], *csr)
    if kind == "resident":
        s.factor()
    return dict(kind=kind, solver=s, B=B, X=torch.zeros_like(B), nrhs=case["nrhs"])


def run(state):
    kind = state["kind"]
    if kind == "host":
        return hs.dspike_core_host(state["A"], state["B"])
    if kind == "band":
        return hs.host_solve(state["A"], state["B"])
    if kind == "batch":
        state["batch"].solve_dev(state["prep"])
        return state["X"]
    if kind == "step":
        state["solver"].factor()
    state["solver"].solve_dev(state["B"], state["X"], state["nrhs"])
    return state["X"]


# ------------------------------------------------------------------------------- accounting

def work(case):
    """Bytes: the CSR matrix and the right-hand sides read once, the solution written once (a resident
    solve also reads its banded factors).  Flops: banded LU, forward and backward substitution and the
    residual of every column."""
    def one(n, kl, ku, fill, m, cplx, resident=False, s=8):
        h, c = (16, 4.0) if cplx else (8, 1.0)
        nnz = n * (1 + (kl + ku) * fill)
        by = nnz * (h + 4) + 4.0 * (n + 1) + 2.0 * n * m * h
        fl = 2.0 * n * (kl + ku) * m + 2.0 * nnz * m
        if resident:
            by += n * (kl + ku + 1.0) * s
        else:
            fl += 2.0 * n * kl * ku
        return by, c * fl
    kind = case["kind"]
    if kind == "batch":
        t = [one(n, k, k, case["fill"], m, False) for n, k, m in _sizes(case)]
        return {"bytes": sum(a for a, _ in t), "flops": sum(b for _, b in t)}
    if kind == "band":
        n, k, m = 2 * case["k"] * case["parts"], case["k"], case["nrhs"]
        w = 3 * k - 1                                                   # bandwidth of the reduced system
        by, _ = one(n, k, k, 1.0, m, False)
        return {"bytes": by, "flops": 2.0 * n * w * w + 4.0 * n * w * m}
    s = (8 if case.get("cplx") else 4) * (2 if case.get("prec", "fp64") == "fp64" else 1)
    by, fl = one(case["n"], case["kl"], case["ku"], case["fill"], case["nrhs"], case.get("cplx", False), kind == "resident", s)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """FP64 factors: measured 2e-16 to 2e-15 from the 64-bit solution.  Mixed precision: measured 2e-14 to
    1e-12 (FP32 factors leave about 1e-7, which one FP64 refinement pass squares), whichever way the sums
    of the factorization are ordered."""
    if case["kind"] in ("host", "band") or case.get("prec") == "fp64":
        return {"rel": 1e-14, "max": 1e-12}
    return {"rel": 5e-12, "max": 5e-10}


# ------------------------------------------------------------------------------- 64-bit solutions

def _jacobi(val, kl, B):
    """Solution of the stacked diagonally dominant systems by Jacobi iteration in 64 bits, to rounding:
    val [rows, width] diagonals, B [rows, m]."""
    rows, width = val.shape
    off = val.t().contiguous()
    dinv = 1.0 / off[kl][:, None]
    X = B * dinv
    for _ in range(400):
        Y = B.clone()
        for d in range(width):
            s = d - kl                                                 # column = row + s
            if s == 0:
                continue
            lo, hi = max(0, -s), min(rows, rows - s)
            Y[lo:hi].addcmul_(off[d, lo:hi, None], X[lo + s:hi + s], value=-1.0)
        Y *= dinv
        step = float((Y - X).abs().max() / Y.abs().max())
        X = Y
        if step < 1e-16:
            break
    return X


def exact(case, seed):
    kind = case["kind"]
    if kind == "band":
        R, B = _reduced(case, seed)
        return np.asfortranarray(np.linalg.solve(R, B))
    if kind == "batch":
        spec, groups, B = _batch(case, seed)
        first = np.concatenate([[0], np.cumsum([n * m for n, _, m in spec])])
        X = torch.empty_like(B)
        for k, ids, (val, _, _) in groups:
            rows, mm = val.shape[0], max(spec[i][2] for i in ids)
            R = torch.zeros(rows, mm, dtype=B.dtype, device=DEV)
            r0 = 0
            for i in ids:
                n, _, m = spec[i]
                R[r0:r0 + n, :m] = B[first[i]:first[i + 1]].view(m, n).t()
                r0 += n
            Y, r0 = _jacobi(val, k, R), 0
            for i in ids:
                n, _, m = spec[i]
                X[first[i]:first[i + 1]] = Y[r0:r0 + n, :m].t().reshape(-1)
                r0 += n
        return X
    val, _, _, B = _single(case, seed)
    X = _jacobi(val, case["kl"], B.t().contiguous()).t().contiguous()
    return np.asfortranarray(X.cpu().numpy().T) if kind == "host" else X
