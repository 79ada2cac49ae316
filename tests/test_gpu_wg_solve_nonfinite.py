"""Batched solves with stored factors whose solution overflows: a zero on U's
diagonal, an infinite right-hand side.  Rows past the order (blocks hold 16)
stay out of it, in both forms (a workgroup per system up to 1024 systems, a
wave per system above).

The off-diagonal entries are all -0.01, so every product with +Inf adds +Inf
and each entry of the exact answer is +Inf; a right-hand side of zeros beside
it stays zero."""
import numpy as np
import pytest
import torch

import tmv_amd

pytestmark = pytest.mark.gpu


def batch(n, count, dtype, LU):
    b = tmv_amd.Batch([n] + [1] * (count - 1), [2] + [1] * (count - 1), dtype=dtype)
    b.A.fill_(1.0)
    b.a(0).copy_(torch.from_numpy(LU))
    b.piv(0).copy_(torch.arange(n))
    return b


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("count", [3, 1030])
@pytest.mark.parametrize("n", [5, 40, 72, 200, 250])
def test_overflow_stays_in_range(dev, dtype, count, n):
    LU = np.full((n, n), -0.01)
    np.fill_diagonal(LU, 2.0)
    singular = LU.copy()
    singular[n - 1, n - 1] = 0.0
    rhs = np.zeros((n, 2))
    rhs[:, 0] = 1.0
    inf_last = np.zeros((n, 2))
    inf_last[n - 1, 0] = np.inf
    for name, M, B, trans in (("zero diagonal", singular, rhs, False),
                              ("zero diagonal", singular, rhs, True),
                              ("infinite entry", LU, inf_last, False)):
        print(f"{name} n {n} count {count} trans {trans} {dtype}", flush=True)
        b = batch(n, count, dtype, M)
        b.b(0).copy_(torch.from_numpy(B))
        tmv_amd.getrs_batched(b, trans=trans)
        X = b.b(0).cpu().numpy()
        assert np.all(np.isposinf(X[:, 0])), (name, trans)
        assert np.all(X[:, 1] == 0), (name, trans)
