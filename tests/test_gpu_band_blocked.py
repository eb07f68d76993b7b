"""The blocked band LU and the register-window band solves (k_gbtrf_blk, k_gbtrs_fwd / _bwd) through
spike_band_solve_host: orders around the panel width (32, complex 16) and the 64-row windows, one-sided
and empty bands, bandwidths at the edges of the register windows, interchanges with rows min(ku, kl) away
and, by the cyclic matrices, with the last row of the lower band, complex bands on both sides of the line
between panels and columns (band_lu_panels), and a band too wide for the panels (kl > 448).

The matrices have singular values >= 1.2 and norms <= 2.8 (a permutation of 2 I inside the band plus
noise with row sums <= 0.8), so after the FP64 refinement the residual is at rounding level: 1e-14,
and the solution agrees with the oracle's band LU within 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hs():
    import hspike_amd
    hspike_amd.load()
    return hspike_amd


def pivoting_band(hs, n, ku, kl, seed, cplx, cyclic=False):
    """2 at (i, s(i)), zero diagonal where s(i) != i; s reverses groups of min(ku, kl) + 1 rows, or, cyclic,
    moves each row of groups of kl + 1 one column up and the group's last row to its first column."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), ku + kl + 1)
    j = i + np.tile(np.arange(-kl, ku + 1), n)
    keep = (j >= 0) & (j < n)
    i, j = i[keep], j[keep]
    v = rng.uniform(-1, 1, i.size) * (0.8 / max(ku + kl, 1))
    if cplx:
        v = v * np.exp(2j * np.pi * rng.uniform(0, 1, i.size))
    m = kl + 1 if cyclic else min(ku, kl) + 1
    first = (i // m) * m
    to = np.where(first + m <= n, np.where(i + 1 < first + m, i + 1, first) if cyclic else 2 * first + m - 1 - i, i)
    v[(j == i) & (to != i)] = 0.0
    v[j == to] = 2.0
    rp = np.zeros(n + 1, dtype=np.int32)
    np.add.at(rp, i + 1, 1)
    return hs.CSRMatrix(n, np.cumsum(rp).astype(np.int32), j.astype(np.int32), v)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n,ku,kl,nrhs", [
    (2, 1, 1, 1), (15, 0, 3, 2), (16, 3, 0, 1), (31, 30, 30, 1), (32, 5, 2, 3), (33, 2, 7, 1), (64, 15, 16, 2), (65, 16, 15, 1),
    (129, 63, 63, 2), (200, 64, 64, 3), (300, 65, 100, 1), (500, 191, 60, 2), (700, 100, 191, 17), (1000, 250, 192, 1),
    (1100, 20, 448, 1), (1200, 10, 460, 2),
])
def test_band_solve_matches_oracle(hs, oracle_mod, n, ku, kl, nrhs, cplx):
    A = pivoting_band(hs, n, ku, kl, seed=n + ku, cplx=cplx)
    B = hs.gen_dense(n, nrhs, seed=3, complex=cplx)
    X, rel = hs.band_solve(A, B)
    assert rel.max() <= 1e-14, rel
    Xo = oracle_mod.direct_solve(oracle_mod.CSR(A.n, A.rowptr, A.colind, A.aij), B)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= 1e-12


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n,ku,kl,nrhs", [
    (2, 1, 1, 1), (33, 2, 7, 1), (65, 16, 31, 2), (97, 1, 32, 1), (200, 64, 64, 3), (300, 65, 100, 1), (700, 100, 191, 3), (1000, 1, 192, 1),
    (1400, 20, 448, 1), (1400, 10, 460, 2),
])
def test_interchanges_with_the_last_row_of_the_band(hs, oracle_mod, n, ku, kl, nrhs, cplx):
    A = pivoting_band(hs, n, ku, kl, seed=n + kl, cplx=cplx, cyclic=True)
    assert (A.rowptr[1:] > A.rowptr[:-1]).all() and abs(A.aij[(A.colind == 0) & (np.repeat(np.arange(n), np.diff(A.rowptr)) == kl)]) == 2.0
    B = hs.gen_dense(n, nrhs, seed=3, complex=cplx)
    X, rel = hs.band_solve(A, B)
    assert rel.max() <= 1e-14, rel
    Xo = oracle_mod.direct_solve(oracle_mod.CSR(A.n, A.rowptr, A.colind, A.aij), B)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= 1e-12


@pytest.mark.parametrize("n,ku,kl,nrhs", [(112, 100, 110, 1), (113, 112, 100, 2), (127, 110, 110, 1), (129, 120, 128, 3), (300, 100, 95, 1),
                                          (300, 95, 90, 1), (700, 448, 31, 1), (640, 300, 448, 1)])
def test_complex_panels(hs, oracle_mod, n, ku, kl, nrhs):
    test_band_solve_matches_oracle(hs, oracle_mod, n, ku, kl, nrhs, True)
    test_interchanges_with_the_last_row_of_the_band(hs, oracle_mod, n, ku, min(kl, n - 1), nrhs, True)


@pytest.mark.parametrize("col", [0, 31, 32, 77, 99])
def test_zero_column_is_singular(hs, col):
    A = pivoting_band(hs, 100, 4, 6, seed=1, cplx=False)
    aij = np.where(A.colind == col, 0.0, A.aij)
    with pytest.raises(hs.SpikeError) as ex:
        hs.band_solve(hs.CSRMatrix(A.n, A.rowptr, A.colind, aij), np.ones((100, 1)))
    assert ex.value.code == -4
    assert "column %d" % col in str(ex.value)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n,ku,row", [(200, 0, 70), (200, 3, 70), (64, 0, 0), (300, 40, 256), (130, 100, 127)])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_nonfinite_right_hand_side_stays_where_it_is_coupled(hs, n, ku, row, cplx, value):
    """Upper triangular bands (kl = 0): the rows below a row with a non-finite right-hand side do not depend on
    it; on a diagonal matrix no other row does."""
    rng = np.random.default_rng(3)
    i = np.repeat(np.arange(n), ku + 1)
    j = i + np.tile(np.arange(ku + 1), n)
    keep = j < n
    v = rng.uniform(-1, 1, i.size) / (ku + 1)
    v[j == i] = 2.0
    rp = np.zeros(n + 1, dtype=np.int32)
    np.add.at(rp, i[keep] + 1, 1)
    A = hs.CSRMatrix(n, np.cumsum(rp).astype(np.int32), j[keep].astype(np.int32), v[keep] + 0j if cplx else v[keep])
    B = hs.gen_dense(n, 1, seed=5, complex=cplx)
    X0, _ = hs.band_solve(A, B)
    B[row] = value
    X, _ = hs.band_solve(A, B)
    assert not np.isfinite(X[row]).any()
    free = np.arange(n) > row if ku else np.arange(n) != row
    assert np.allclose(X[free], X0[free], rtol=1e-13, atol=1e-13)
