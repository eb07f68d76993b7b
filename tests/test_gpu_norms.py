"""Sums of the residual norms over slabs of chunks (systems of more than 8192 chunks of 64 rows): orders
on both sides of the line, and in one batch with a small system.  The reported residual against a CPU
residual of the returned solution, on a solve stopped after its first mixed-precision pass (there the
residual is about 1e-7 and rounding, 1e-15, cannot matter): 1e-6 relative.  Alone equals in the batch,
bit for bit."""
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
