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


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("count", [3, 1030])
@pytest.mark.parametrize("n", [5, 40, 72, 200, 250])
def test_zero_entry_takes_no_part(dev, dtype, count, n):
    """A zero entry is skipped by the substitution: what the factors hold in
    its column does not matter, Inf and NaN included."""
    g = np.random.default_rng(n)
    LU = g.uniform(-1, 1, (n, n)) + n * np.eye(n)
    rhs = np.zeros((n, 2))
    rhs[n // 2, :] = (1.0, -2.0)
    want = LU.copy()                # column n - 1: x there is zero, L's columns
    LU[: n - 1, n - 1] = np.inf     # before n / 2: so is y
    LU[1:, 0] = np.nan
    want[n // 2 + 1:, n // 2] = LU[n // 2 + 1:, n // 2] = 0.0
    print(f"zero entries n {n} count {count} {dtype}", flush=True)
    b = batch(n, count, dtype, LU)
    b.b(0).copy_(torch.from_numpy(rhs))
    tmv_amd.getrs_batched(b)
    U = np.triu(want)[: n // 2 + 1, : n // 2 + 1]
    x = np.linalg.solve(U, rhs[: n // 2 + 1])
    X = b.b(0).cpu().numpy()
    eps = np.finfo(np.float64 if dtype == torch.float64 else np.float32).eps
    assert np.all(X[n // 2 + 1:] == 0)
    assert np.allclose(X[: n // 2 + 1], x, rtol=8 * n * eps, atol=8 * n * eps * np.abs(x).max())
