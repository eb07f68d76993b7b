"""The block-Jacobi sweep of the reduced system (k_red_jacobi): every block size, unequal tips whose
bounds fall inside a 16-row tile, one to four column tiles per workgroup and a remainder, a single
interface (no neighbours) and several; complex systems through their solution.

xr against the oracle's direct solve of the reference's R: both are FP64 solutions of a well
conditioned system from tips that agree to 1e-10, so 1e-9 relative bounds the difference; the
full solution of the same dominant systems likewise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hs():
    import hspike_amd
    hspike_amd.load()
    return hspike_amd


@pytest.mark.parametrize("nrhs", [1, 17, 40, 64])
@pytest.mark.parametrize("ku,kl,P", [(1, 3, 2), (16, 9, 5), (17, 32, 3), (5, 40, 4), (64, 33, 2), (65, 128, 3), (120, 7, 4),
                                     (129, 200, 2)])
def test_reduced_solution_matches_oracle(hs, oracle_mod, ku, kl, P, nrhs):
    b = next(x for x in (16, 32, 64, 128, 256) if max(ku, kl) <= x)
    n = P * (2 * b + 5) + 3
    A = hs.gen_banded(n, ku, kl, fill=0.4, dom=(1.1, 1.1), diag_floor=1.0, seed=ku + kl)
    B = hs.gen_dense(n, nrhs, seed=nrhs)
    s = hs.Solver("fp64", partitions=P)
    s.set_matrix(A)
    X = s.solve(B)
    st = s.stats()
    assert st["P"] == P and st["reduced_direct"] == 0
    Xo, info = oracle_mod.spike_solve(oracle_mod.CSR(A.n, A.rowptr, A.colind, A.aij), B, P)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= 1e-9
    if st["refine_iters"] == 0:
        xr = s.reduced_solution()
        assert np.linalg.norm(xr - info["xr"]) / np.linalg.norm(info["xr"]) <= 1e-9
    s.close()


@pytest.mark.parametrize("k,P,nrhs", [(3, 3, 1), (3, 4, 33), (20, 4, 17), (20, 3, 40), (30, 4, 64), (40, 3, 5), (40, 2, 33), (90, 2, 20), (140, 2, 3)])
def test_complex_reduced(hs, oracle_mod, k, P, nrhs):
    b = next(x for x in (16, 32, 64, 128, 256) if k <= x)
    n = P * (2 * b + 5) + 3
    A = hs.gen_banded(n, k, k, fill=0.4, dom=(1.2, 1.2), diag_floor=1.0, seed=k, complex=True)
    B = hs.gen_dense(n, nrhs, seed=nrhs, complex=True)
    s = hs.Solver("fp64", partitions=P)
    s.set_matrix(A)
    X = s.solve(B)
    assert s.stats()["reduced_direct"] == 0
    Xo = oracle_mod.direct_solve(oracle_mod.CSR(A.n, A.rowptr, A.colind, A.aij), B)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) <= 1e-9
    s.close()
