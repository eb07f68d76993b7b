"""The wide factor (b = 256, and complex FP64 at b = 128): pivot tiles that are dominant by rows (the
in-register inversion), tiles that need interchanges over all 16 rows (the LDS one), and mixes of both
in one matrix; unequal bandwidths, so tiles without entries of B_j and C_j are skipped; last blocks of
16 and 17 rows, of one row, and whole ones.

The matrices are a permutation of 2 I inside 16-row groups (or 2 I) plus band noise with row sums at
most 0.8: singular values are at least 1.2, so against the oracle's band LU the FP64 solution differs
by a small multiple of the rounding (1e-11) and the mixed one, at a residual of 1e-10, by 2.4e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hs():
    import hspike_amd
    hspike_amd.load()
    return hspike_amd


def reversed_band(hs, n, ku, kl, group, rows_from, cplx, seed):
    """2 at (i, s(i)): s reverses groups of `group` rows from row rows_from on, the identity before."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), ku + kl + 1)
    j = i + np.tile(np.arange(-kl, ku + 1), n)
    keep = (j >= 0) & (j < n)
    i, j = i[keep], j[keep]
    v = 0.8 / (ku + kl + 1) * rng.uniform(-1, 1, i.size)
    if cplx:
        v = v * np.exp(2j * np.pi * rng.uniform(0, 1, i.size))
    first = (i // group) * group
    to = np.where((i >= rows_from) & (first + group <= n), 2 * first + group - 1 - i, i)
    v[(j == i) & (to != i)] = 0.0
    v[j == to] = 2.0
    rp = np.zeros(n + 1, dtype=np.int32)
    np.add.at(rp, i + 1, 1)
    return hs.CSRMatrix(n, np.cumsum(rp).astype(np.int32), j.astype(np.int32), v)


@pytest.mark.parametrize("ku,kl,prec,cplx", [(200, 140, "mixed", False), (130, 256, "mixed", False), (150, 190, "fp64", False),
                                             (140, 160, "mixed", True), (100, 128, "fp64", True)])
@pytest.mark.parametrize("group,frac", [(1, 1.0), (16, 0.0), (16, 0.5)])
@pytest.mark.parametrize("rest", [16, 0])
def test_wide_factor_matches_oracle(hs, oracle_mod, ku, kl, prec, cplx, group, frac, rest):
    b = 128 if max(ku, kl) <= 128 else 256
    part = 2 * b + rest                          # partitions start on multiples of 16, the last has one row more
    n = 2 * part + 1
    A = reversed_band(hs, n, ku, kl, group, int(frac * n) // 16 * 16, cplx, seed=ku)
    B = hs.gen_dense(n, 2, seed=5, complex=cplx)
    s = hs.Solver(prec, partitions=2)
    s.set_matrix(A)
    X = s.solve(B)
    assert s.stats()["b"] == b
    assert hs.residual(A, X, B).max() <= 1e-10
    Xo = oracle_mod.direct_solve(oracle_mod.CSR(A.n, A.rowptr, A.colind, A.aij), B)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= (1e-11 if prec == "fp64" else 2.4e-10)
    s.close()
