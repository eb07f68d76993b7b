"""The dense-tile residual (k_residual_mm) through whole solves: orders around its 64-row chunks and
16-row tiles (test_small_orders_with_the_dense_tile where few columns leave them to the gather kernel),
one-sided bands, one to four column tiles with odd counts, rows stored in any column order and split
entries (duplicates are summed), bands with five entries per row, in a batch that mixes systems of both
residual kernels.

The solver's reported residual against a CPU residual (numpy, FP64) of the returned solution: both
are rounding-level quantities of the same solution, so they are compared on a solve stopped after its
first mixed-precision pass, where the residual is about 1e-7 and rounding (1e-15) cannot matter: 1e-6
relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hs():
    import hspike_amd
    hspike_amd.load()
    return hspike_amd


def cpu_relres(A, X, B):
    R = B - A.to_scipy() @ X
    return np.linalg.norm(R, axis=0) / np.linalg.norm(B, axis=0)


def shuffled(hs, A, seed):
    """Rows stored in random column order."""
    rng = np.random.default_rng(seed)
    perm = np.concatenate([rng.permutation(np.arange(a, b)) for a, b in zip(A.rowptr[:-1], A.rowptr[1:])])
    return hs.CSRMatrix(A.n, A.rowptr, A.colind[perm], A.aij[perm])


@pytest.mark.parametrize("n,ku,kl,nrhs", [(63, 2, 2, 1), (64, 5, 1, 3), (65, 0, 4, 2), (200, 16, 0, 17), (1000, 30, 32, 9), (777, 7, 20, 33),
                                          (1300, 64, 40, 16), (1201, 33, 64, 64), (2500, 128, 70, 35), (2100, 100, 128, 64)])
def test_reported_residual(hs, n, ku, kl, nrhs):
    A = shuffled(hs, hs.gen_banded(n, ku, kl, fill=0.6, dom=(1.1, 1.1), diag_floor=1.0, seed=n), n)
    B = hs.gen_dense(n, nrhs, seed=2)
    s = hs.Solver("mixed", max_refine=0, tol=1e-3)
    s.set_matrix(A)
    X = s.solve(B)
    got = s.stats()["max_rel_residual"]
    ref = cpu_relres(A, X, B).max()
    assert abs(got - ref) <= 1e-6 * ref + 1e-15
    t = hs.Solver("mixed")
    t.set_matrix(A)
    assert cpu_relres(A, t.solve(B), B).max() <= 1e-10
    s.close()
    t.close()


@pytest.mark.parametrize("n,ku,kl,nrhs", [(63, 2, 2, 9), (65, 0, 4, 10), (64, 3, 0, 9), (1, 0, 0, 9), (17, 1, 1, 64)])
def test_small_orders_with_the_dense_tile(hs, n, ku, kl, nrhs):
    """More than 8 columns: at b = 16 the dense tile whatever the entries per row."""
    test_reported_residual(hs, n, ku, kl, nrhs)


@pytest.mark.parametrize("k,nrhs", [(7, 1), (7, 4), (7, 16), (30, 3), (30, 9), (61, 8), (61, 16), (61, 33), (128, 17), (128, 64)])
def test_stencil(hs, k, nrhs):
    """Five-point Laplacian on a grid of width k, 5 entries per row: both residual kernels, by the columns."""
    n = 9 * k + 4
    off = np.array([-k, -1, 0, 1, k])
    i = np.repeat(np.arange(n), 5)
    j = i + np.tile(off, n)
    v = np.tile([-1.0, -1.0, 4.5, -1.0, -1.0], n)
    keep = (j >= 0) & (j < n)
    rp = np.zeros(n + 1, dtype=np.int32)
    np.add.at(rp, i[keep] + 1, 1)
    A = hs.CSRMatrix(n, np.cumsum(rp).astype(np.int32), j[keep].astype(np.int32), v[keep])
    B = hs.gen_dense(n, nrhs, seed=4)
    s = hs.Solver("mixed", max_refine=0, tol=1e-3)
    s.set_matrix(A)
    X = s.solve(B)
    got, ref = s.stats()["max_rel_residual"], cpu_relres(A, X, B).max()
    assert abs(got - ref) <= 1e-6 * ref + 1e-15
    s.close()


def test_duplicate_entries_are_summed(hs):
    """Entry (r, r) split in two halves: the factorization keeps one of them, the residual sums both, so
    the solve ends unconverged instead of with a wrong answer."""
    n = 300
    A = hs.gen_banded(n, 3, 3, fill=1.0, dom=(1.2, 1.2), diag_floor=1.0, seed=1)
    r, q = 150, int(A.rowptr[150]) + 3
    assert A.colind[q] == r
    aij = A.aij.copy()
    aij[q] *= 0.5
    D = hs.CSRMatrix(n, A.rowptr + (np.arange(n + 1) > r), np.insert(A.colind, q, r), np.insert(aij, q, aij[q]))
    B = hs.gen_dense(n, 2, seed=3)
    s = hs.Solver("fp64", partitions=1, max_refine=0)
    s.set_matrix(D)
    X = s.solve(B, allow_unconverged=True)
    got, ref = s.stats()["max_rel_residual"], cpu_relres(A, X, B).max()
    assert ref > 1e-3 and abs(got - ref) <= 1e-10
    s.close()


def test_mixed_batch_equals_alone(hs):
    import torch
    dev = torch.device("cuda:0")
    systems = []
    for i, (n, k, fill, nrhs) in enumerate([(900, 40, 0.1, 2), (900, 40, 0.9, 2), (1500, 60, 0.1, 16), (700, 3, 1.0, 5), (2000, 100, 0.2, 40),
                                            (2000, 100, 0.2, 3)]):
        A = hs.gen_banded(n, k, k, fill=fill, dom=(1.1, 1.1), diag_floor=1.0, seed=60 + i)
        B = hs.gen_dense(n, nrhs, seed=70 + i)
        systems.append(dict(n=n, nrhs=nrhs, rowptr=torch.from_numpy(A.rowptr).to(dev), colind=torch.from_numpy(A.colind).to(dev),
                            aij=torch.from_numpy(A.aij).to(dev), b=torch.from_numpy(np.ascontiguousarray(B.T)).to(dev),
                            x=torch.zeros((nrhs, n), dtype=torch.float64, device=dev)))
    rel, _ = hs.Batch("mixed").solve_dev(systems)
    torch.cuda.synchronize()
    assert rel.max() <= 1e-10
    for q, s in enumerate(systems):
        alone = dict(s, x=torch.zeros_like(s["x"]))
        r1, _ = hs.Batch("mixed").solve_dev([alone])
        torch.cuda.synchronize()
        assert torch.equal(alone["x"], s["x"]) and r1[0] == rel[q]
