"""A batch of several block sizes with graph = 1: each block size's launches run on a stream of their
own, in the factorization and in the replayed solve.  Repeated work with new values must give the eager
batch's bits every time (the tolerance is zero: the same kernels run on the same systems)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,ks", [("mixed", [3, 20, 60, 100, 150]), ("fp64", [150, 3, 100, 20]), ("mixed", [3, 60])])
def test_groups_side_by_side(prec, ks):
    import torch
    import hspike_amd as hs
    hs.load()
    dev = torch.device("cuda:0")
    systems = []
    for i, k in enumerate(ks + ks[:1]):
        n = 9 * max(k, 16) * (4 - i % 3) + i
        A = hs.gen_banded(n, k, k, fill=0.4, dom=(1.2, 1.2), diag_floor=1.0, seed=40 + i)
        B = hs.gen_dense(n, 1 + 5 * i, seed=50 + i)
        systems.append(dict(n=n, nrhs=1 + 5 * i, rowptr=torch.from_numpy(A.rowptr).to(dev), colind=torch.from_numpy(A.colind).to(dev),
                            aij=torch.from_numpy(A.aij).to(dev), b=torch.from_numpy(np.ascontiguousarray(B.T)).to(dev)))
    sel = [dict(s, x=torch.zeros_like(s["b"])) for s in systems]
    ser = [dict(s, x=torch.zeros_like(s["b"])) for s in systems]
    bt, ref = hs.Batch(prec, graph=True), hs.Batch(prec)
    replays = 0
    for step in range(5):
        for s in systems:
            s["aij"].mul_(1.0 + 0.25 * step)                # both batches read the same arrays
        torch.cuda.synchronize()
        _, st = bt.solve_dev(sel)
        replays += st["graph_replayed"]
        ref.solve_dev(ser)
        torch.cuda.synchronize()
        for a, b in zip(sel, ser):
            assert torch.equal(a["x"], b["x"]), (step, a["n"])
            assert torch.isfinite(a["x"]).all()
        assert st["ms_factor"] > 0
    assert replays >= 2
    bt.close()
    ref.close()
