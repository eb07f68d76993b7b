"""Pivot reciprocals, through the solution of diagonal systems with right-hand sides of ones: one block inverse,
one product with 1 and exact zeros.

FP64: the correctly rounded reciprocal, as numpy gives it, over the exponents and at the edges of the mantissa (all ones and its neighbours, where two Newton steps from a hardware seed are not enough).
Complex: Smith's form with correctly rounded divisions, whose error over |1/d| is 0.653 units (2^-53, FP32
factors 2^-24) root mean square and below 2.5 over numbers with parts in (-1, 1); 2 10^5 samples move the root
mean square by less than 0.5%, so 0.67 separates it from a form with one more rounding per part (0.78)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reciprocals(prec, d):
    import torch
    import hspike_amd as hs
    hs.load()
    n, dev = d.size, torch.device("cuda:0")
    rp = torch.arange(n + 1, dtype=torch.int32, device=dev)
    v = torch.from_numpy(d).to(dev)
    b = torch.ones(1, n, dtype=v.dtype, device=dev)
    x = torch.zeros_like(b)
    s = hs.Solver(prec, max_refine=0, tol=1.0)
    s.set_matrix_dev(n, rp, rp[:n].contiguous(), v)
    s.factor()
    s.solve_dev(b, x, 1)
    torch.cuda.synchronize()
    s.close()
    return x[0].cpu().numpy()


@pytest.mark.parametrize("lo,hi", [(0, 1), (-30, 30), (-1000, 1000), (1015, 1023), (-1021, -1015)])
def test_fp64_reciprocal_is_the_division(lo, hi):
    rng = np.random.default_rng(lo & 0xFFFF)
    n = 1 << 20
    m = 1.0 + rng.uniform(0, 1, n)
    edge = np.concatenate([1.0 + np.arange(64) * 2.0 ** -52, 2.0 - np.arange(1, 65) * 2.0 ** -52, 1.5 + np.arange(-64, 64) * 2.0 ** -52])
    m[:edge.size] = edge
    m = np.minimum(m, 2.0 - 2.0 ** -52)
    d = np.ldexp(m, rng.integers(lo, hi, n)) * rng.choice([-1.0, 1.0], n)
    assert np.array_equal(reciprocals("fp64", d), 1.0 / d)


@pytest.mark.parametrize("prec,u", [("fp64", 2.0 ** -53), ("mixed", 2.0 ** -24)])
@pytest.mark.parametrize("exp", [0, 40, -40])
def test_complex_reciprocal_error(prec, u, exp):
    rng = np.random.default_rng(exp + 100)
    n = 200_000
    d = (rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)).astype(np.complex64 if prec == "mixed" else np.complex128)
    d = d.astype(np.complex128) * 2.0 ** exp
    ref = 1 / d.astype(np.clongdouble)
    err = np.abs((reciprocals(prec, d) - ref) / ref).astype(np.float64) / u
    assert err.max() <= 2.5 and np.sqrt((err ** 2).mean()) <= 0.67
