"""Sums of the residual norms over slabs of chunks (systems of more than 8192 chunks of 64 rows): orders
on both sides of the line, and in one batch with a small system.  The reported residual against a CPU
residual of the returned solution, on a solve stopped after its first mixed-precision pass (there the
residual is about 1e-7 and rounding, 1e-15, cannot matter): 1e-6 relative.  Alone equals in the batch,
bit for bit, wherever the large systems stand in it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs", [(8192 * 64, 3), (8192 * 64 + 1, 3), (8193 * 64 + 17, 1), (600_001, 64), (8320 * 64, 5)])
def test_norms_around_the_line(n, nrhs):
    import torch
    import hspike_amd as hs
    hs.load()
    dev = torch.device("cuda:0")
    lst = []
    for i, (nn, m) in enumerate([(n, nrhs), (700, 2)]):
        A = hs.gen_banded(nn, 3, 3, fill=0.8, dom=(1.1, 1.1), diag_floor=1.0, seed=5 + i)
        B = hs.gen_dense(nn, m, seed=7 + i)
        d = dict(n=nn, nrhs=m, rowptr=torch.from_numpy(A.rowptr).to(dev), colind=torch.from_numpy(A.colind).to(dev),
                 aij=torch.from_numpy(A.aij).to(dev), b=torch.from_numpy(np.ascontiguousarray(B.T)).to(dev))
        d["x"] = torch.zeros_like(d["b"])
        lst.append((d, A, B))
    bt = hs.Batch("mixed", max_refine=0, tol=1e-3)
    rel, _ = bt.solve_dev([d for d, _, _ in lst])
    for i, (d, A, B) in enumerate(lst):
        X = d["x"].cpu().numpy().T
        ref = (np.linalg.norm(B - A.to_scipy() @ X, axis=0) / np.linalg.norm(B, axis=0)).max()
        assert abs(rel[i] - ref) <= 1e-6 * ref + 1e-15
    alone = dict(lst[0][0], x=torch.zeros_like(lst[0][0]["b"]))
    rel1, _ = bt.solve_dev([alone])
    assert rel1[0] == rel[0] and torch.equal(alone["x"], lst[0][0]["x"])
    bt.close()


def device_system(torch, hs, n, nrhs, seed, A=None):
    dev = torch.device("cuda:0")
    A = A or hs.gen_banded(n, 3, 3, fill=0.8, dom=(1.1, 1.1), diag_floor=1.0, seed=seed)
    B = hs.gen_dense(n, nrhs, seed=seed + 1)
    d = dict(n=n, nrhs=nrhs, rowptr=torch.from_numpy(A.rowptr).to(dev), colind=torch.from_numpy(A.colind).to(dev),
             aij=torch.from_numpy(A.aij).to(dev), b=torch.from_numpy(np.ascontiguousarray(B.T)).to(dev))
    return dict(d, x=torch.zeros_like(d["b"]))


def test_large_systems_among_small_ones():
    """Two systems above the line among small ones and one at the line: each one's residual is the one it
    gets alone, bit for bit, eager and replayed."""
    import torch
    import hspike_amd as hs
    hs.load()
    lst = [device_system(torch, hs, n, m, 20 + i) for i, (n, m) in
           enumerate([(900, 2), (8200 * 64, 2), (1300, 5), (8192 * 64, 1), (8193 * 64, 3), (64, 1)])]
    bt = hs.Batch("mixed", tol=1e-3, max_refine=0, graph=True)
    rels = [bt.solve_dev(lst)[0].copy() for _ in range(3)]
    for q, s in enumerate(lst):
        alone, _ = hs.Batch("mixed", tol=1e-3, max_refine=0).solve_dev([dict(s, x=torch.zeros_like(s["x"]))])
        assert all(r[q] == alone[0] for r in rels), q
    bt.close()


def test_small_systems_pay_nothing_for_a_large_one():
    """Time of the norm sums of 4096 small systems and a large one, against 4096 small ones and the large one
    alone: the slabs of the large one add little (27 us; 141 us when every system had slabs)."""
    import torch
    import hspike_amd as hs
    hs.load()
    small, big = device_system(torch, hs, 1500, 4, 40), device_system(torch, hs, 8200 * 64, 4, 50)
    many = [dict(small, x=torch.zeros_like(small["x"])) for _ in range(4096)]

    def norms(systems):
        bt = hs.Batch("mixed", tol=1e-3, max_refine=0)
        prep, best = bt.prepare(systems), 1e9
        for _ in range(8):
            best = min(best, bt.solve_dev(prep)[1]["ms_norms"])
        bt.close()
        return best

    assert norms([big] + many) <= 2.0 * (norms(many) + norms([big]))
