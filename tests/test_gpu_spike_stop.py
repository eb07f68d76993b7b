"""Spike sweeps that stop at different blocks in the items of one partition: the W columns of a partition
of b = 128 (or FP64 / complex b = 64) are swept by several workgroups, each of which stops at its own decay
and leaves zeros behind it.  The first factorization fills the spike storage with slowly decaying
columns; the second, on the same handle, has fast ones, slow ones and empty ones side by side, so a
block that is neither computed nor cleared would show.  The solution against the oracle's band solve
(FP64; the matrices' condition numbers are below 100): 1e-11 relative."""
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
