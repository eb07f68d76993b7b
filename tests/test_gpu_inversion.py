"""The block inversion of the factor (16-wide panels, each pivot tile inverted by one wave over 4x4
pivot blocks): every block size of the register kernels, every position of an interchange inside
a 4x4 pivot block, partial last blocks, and dominant blocks (which take no interchange).

The matrices are a permutation of 2 I inside 4x4 blocks (or 2 I) plus band noise with row sums at
most 0.8, so singular values are at least 1.2 and the FP64 solve's error against the oracle's band
LU is a small multiple of the rounding: 1e-11; mixed precision ends at a residual of 1e-10, so its
error is at most 1e-10 ||b|| / 1.2 against ||x|| >= ||b|| / 2.8: 2.4e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hs():
    import hspike_amd
    hspike_amd.load()
    return hspike_amd


def permuted_band(hs, n, k, flip, cplx, seed):
    """2 at (i, i ^ flip) where that stays inside the matrix (else at (i, i)), noise elsewhere."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), 2 * k + 1)
    j = i + np.tile(np.arange(-k, k + 1), n)
    keep = (j >= 0) & (j < n)
    i, j = i[keep], j[keep]
    v = 0.8 / (2 * k + 1) * rng.uniform(-1, 1, i.size)
    if cplx:
        v = v * np.exp(2j * np.pi * rng.uniform(0, 1, i.size))
    whole = (i // 4) * 4 + 4 <= n
    to = np.where(whole, i ^ flip, i)
    v[(j == i) & (to != i)] = 0.0
    v[j == to] = 2.0
    rp = np.zeros(n + 1, dtype=np.int32)
    np.add.at(rp, i + 1, 1)
    return hs.CSRMatrix(n, np.cumsum(rp).astype(np.int32), j.astype(np.int32), v)


@pytest.mark.parametrize("flip", [0, 1, 2, 3])
@pytest.mark.parametrize("k,prec,cplx", [
    (4, "mixed", False), (16, "fp64", False), (16, "mixed", True), (4, "fp64", True), (32, "mixed", False),
    (20, "fp64", False), (32, "mixed", True), (64, "mixed", False), (50, "fp64", False), (64, "mixed", True),
    (40, "fp64", True), (128, "mixed", False), (100, "fp64", False), (70, "mixed", True),
])
def test_inversion_matches_oracle(hs, oracle_mod, k, prec, cplx, flip):
    b = 16 if k <= 16 else (32 if k <= 32 else (64 if k <= 64 else 128))
    n = 3 * (4 * b + 20) + 1                    # P = 3: bounds on multiples of 4, partial last blocks
    A = permuted_band(hs, n, k, flip, cplx, seed=k + flip)
    B = hs.gen_dense(n, 3, seed=2, complex=cplx)
    s = hs.Solver(prec, partitions=3)
    s.set_matrix(A)
    X = s.solve(B)
    st = s.stats()
    assert st["b"] == b and st["P"] == 3
    assert hs.residual(A, X, B).max() <= 1e-10
    Xo = oracle_mod.direct_solve(oracle_mod.CSR(A.n, A.rowptr, A.colind, A.aij), B)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= (1e-11 if prec == "fp64" else 2.4e-10)
    s.close()
