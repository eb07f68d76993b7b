"""Spike sweeps that stop at different blocks in the items of one partition: the W columns of a partition
of b = 128 (or FP64 / complex b = 64) are swept by several workgroups, each of which stops at its own decay
and leaves zeros behind it.  The first factorization fills the spike storage with slowly decaying
columns; the second, on the same handle, has fast ones, slow ones and empty ones side by side
(test_items_stop_apart: in every item; test_fast_and_slow_items: the first half of the columns against the
second, whose stops are computed on the CPU too), so a block that is neither computed nor cleared would show.
The solution against the oracle's band solve (the matrices' condition numbers are about 100 at most; FP64, and
mixed precision, whose last correction leaves its residual far below the tolerance): 1e-11 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,k,cplx", [("mixed", 128, False), ("fp64", 128, False), ("mixed", 100, False), ("fp64", 64, False),
                                         ("fp64", 50, False), ("mixed", 64, True), ("mixed", 33, True)])
@pytest.mark.parametrize("nparts", [2, 3])
def test_items_stop_apart(oracle_mod, prec, k, cplx, nparts):
    import hspike_amd as hs
    hs.load()
    b = 128 if k > 64 else 64
    n = nparts * 24 * b + 5
    rng = np.random.default_rng(k + nparts)
    A = hs.gen_banded(n, k, k, fill=0.2, dom=(1.02, 1.02), diag_floor=1.0, seed=k, **({"complex": True} if cplx else {}))
    rows = np.repeat(np.arange(n), np.diff(A.rowptr))
    B = rng.standard_normal((n, 5)) + (1j * rng.standard_normal((n, 5)) if cplx else 0)
    s = hs.Solver(prec, partitions=nparts)
    s.set_matrix(A)
    X = s.solve(B)
    off = A.colind != rows
    for trial in range(2):
        # off-diagonal columns by their place in a period: cleared, scaled down (a fast decay), kept
        place = (A.colind + 17 * trial) % 96
        aij = np.where(off & (place < 32), 0.0, np.where(off & (place < 64), 1e-4 * A.aij, A.aij))
        M = hs.CSRMatrix(n, A.rowptr, A.colind, aij)
        s.set_matrix(M)
        X = s.solve(B)
        Xo = oracle_mod.direct_solve(oracle_mod.CSR(n, A.rowptr, A.colind, aij), B)
        assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= 1e-11, trial
    s.close()


def forward_stops(D, b, r0, ni, halves):
    """First block j with max |w_j| <= 2^-70 max |w_0| over each set of W columns, w the block forward sweep
    of the partition's coupling columns (None: runs to the end)."""
    nb = ni // b
    blk = lambda i, j: D[r0 + i * b:r0 + (i + 1) * b, r0 + j * b:r0 + (j + 1) * b].toarray()
    S, w, tops = blk(0, 0), D[r0:r0 + b, r0 - b:r0].toarray(), []
    for j in range(nb):
        w = np.linalg.solve(S, w)
        tops.append([np.abs(w[:, h]).max() for h in halves])
        if j + 1 < nb:
            C = blk(j + 1, j)
            S, w = blk(j + 1, j + 1) - C @ np.linalg.solve(S, blk(j, j + 1)), -C @ w
    tops = np.array(tops)
    return [next((j for j in range(1, nb) if t[j] <= 2.0 ** -70 * t[0]), None) for t in tops.T]


@pytest.mark.parametrize("prec,b,cplx", [("mixed", 128, False), ("fp64", 128, False), ("fp64", 64, False), ("mixed", 64, True)])
def test_fast_and_slow_items(oracle_mod, prec, b, cplx):
    """Rows and columns in two classes by their place in the block (first or second half), no entries between
    them: the spike columns of the fast class decay within a few blocks, those of the slow one (averaging rows,
    dominance 1.02) do not, and an item of the sweep holds columns of one class only."""
    import scipy.sparse as sp
    import hspike_amd as hs
    hs.load()
    nparts, nb = 2, 16
    n = nparts * nb * b
    A = hs.gen_banded(n, b, b, fill=0.2, dom=(1.02, 1.02), diag_floor=1.0, seed=b)
    rows = np.repeat(np.arange(n), np.diff(A.rowptr))
    off = A.colind != rows
    same = (rows % b < b // 2) == (A.colind % b < b // 2)

    def matrix(fast):                                        # fast: the rows with entries scaled down
        v = np.where(off, -np.abs(A.aij), 0.0) * np.where(same, 1.0, 0.0) * np.where(fast[rows], 1e-4, 1.0)
        d = np.bincount(rows, weights=np.abs(v), minlength=n)
        d = np.where(fast, np.maximum(d / 1e-4, 1.0), np.maximum(d, 1e-3)) * 1.02
        v = np.where(off, v, d[rows])
        return hs.CSRMatrix(n, A.rowptr, A.colind, v.astype(complex) if cplx else v)

    rng = np.random.default_rng(b)
    B = rng.standard_normal((n, 3)) + (1j * rng.standard_normal((n, 3)) if cplx else 0)
    s = hs.Solver(prec, partitions=nparts, tol=1e-13 if prec == "mixed" else 1e-10)
    s.set_matrix(matrix(np.zeros(n, bool)))
    s.solve(B)
    first = np.arange(n) % b < b // 2
    for fast in (first, ~first):
        M = matrix(fast)
        D = sp.csr_matrix((np.real(M.aij), M.colind, M.rowptr), shape=(n, n))
        stops = forward_stops(D, b, nb * b, nb * b, [slice(0, b // 2), slice(b // 2, b)])
        quick, slow = stops if fast[0] else stops[::-1]
        assert quick is not None and quick < 8 and slow is None, stops
        s.set_matrix(M)
        X = s.solve(B)
        Xo = oracle_mod.direct_solve(oracle_mod.CSR(n, M.rowptr, M.colind, M.aij), B)
        assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= 1e-11
    s.close()


@pytest.mark.parametrize("prec,ku", [("mixed", 2), ("mixed", 60), ("mixed", 140), ("fp64", 2), ("fp64", 140)])
def test_overflowing_spike_is_not_taken_for_a_decayed_one(prec, ku):
    """Two chains in one matrix, even and odd rows: the even W column grows until it overflows in block 2 and is
    NaN from there on, the odd one decays to zero.  The bottom tip of the even column must not be finite (a
    maximum that drops NaN ends the chain there and leaves a tip of zeros)."""
    import hspike_amd as hs
    hs.load()
    b = next(x for x in (16, 32, 64, 128, 256) if ku <= x)
    n = 2 * 7 * b
    g = (1e13 if prec == "mixed" else 1e110) ** (2.0 / b)
    i = np.arange(2, n)
    rows = np.concatenate([np.arange(n), i, [0]])
    cols = np.concatenate([np.arange(n), i - 2, [ku]])
    vals = np.concatenate([np.ones(n), np.where(i % 2 == 0, -g, -0.5), [1e-30]])
    order = np.lexsort((cols, rows))
    rp = np.zeros(n + 1, dtype=np.int32)
    np.add.at(rp, rows + 1, 1)
    A = hs.CSRMatrix(n, np.cumsum(rp).astype(np.int32), cols[order].astype(np.int32), vals[order])
    B = np.zeros((n, 1))
    B[1] = 1.0
    s = hs.Solver(prec, partitions=2, max_refine=0, reduced_solver="jacobi")
    s.set_matrix(A)
    s.solve(B, allow_unconverged=True)
    Wb = s.tips()["Wb"][1]
    assert s.stats()["b"] == b and not np.isfinite(Wb[:, 0]).any(), Wb
    s.close()
