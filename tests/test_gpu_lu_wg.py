"""Batched LU of medium systems (128 < n <= 1024, a workgroup each) against
the oracle: sizes at the edges of its panels, column chunks and workgroup
classes, exact ties, a zero column and a zero matrix.

Bar: pivots identical where the pivot gap exceeds 64 n eps, ||P A - L U||
<= 8 n eps ||A||; ties (a Hadamard matrix, exact in floating point) and the
underflow rule exactly as the oracle."""
import numpy as np
import pytest
import scipy.linalg
import torch

import tmv_amd
from checks import EPS64, EPS32, lu_residual
from tmv_amd import rng

pytestmark = pytest.mark.gpu
SEED = 0x7A15EED


def factor(mats, dtype):
    b = tmv_amd.Batch([len(A) for A in mats], dtype=dtype)
    for i, A in enumerate(mats):
        b.a(i).copy_(torch.from_numpy(A).to(dtype))
    info = tmv_amd.getrf_batched(b).cpu().numpy()
    return b, info


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("ns", [[129, 160, 161, 255, 256], [257, 288, 289, 511, 512, 140],
                                [513, 800, 1023, 1024, 200]])
def test_medium_lu(orc, dev, dtype, ns):
    print(f"medium LU {dtype} {ns}", flush=True)
    eps = EPS64 if dtype == torch.float64 else EPS32
    mats = [rng.uniform_matrix(SEED + n, n, n) for n in ns]
    if dtype == torch.float32:
        mats = [A.astype(np.float32).astype(np.float64) for A in mats]
    b, info = factor(mats, dtype)
    for i, (n, A) in enumerate(zip(ns, mats)):
        assert info[i] == 0
        P = b.piv(i).cpu().numpy()
        _, Po, gaps = orc.getrf(A, gaps=True)
        ok = gaps > 64 * n * eps
        k0 = n if ok.all() else int(np.argmin(ok))
        assert np.array_equal(P[:k0], Po[:k0]), (n, k0)
        assert lu_residual(A, b.a(i).cpu().numpy(), P) <= 8 * n * eps, n


def test_medium_lu_ties_and_zero_columns(orc, dev):
    n = 256
    H = scipy.linalg.hadamard(n).astype(np.float64)
    Z = rng.uniform_matrix(SEED + 1, n, n)
    Z[:, 37] = 0.0
    Z[:, 200] = 0.0
    b, info = factor([H, Z, np.zeros((n, n))], torch.float64)
    LUo, Po = orc.getrf(H)
    assert info[0] == 0
    assert np.array_equal(b.piv(0).cpu().numpy(), Po)
    assert np.array_equal(b.a(0).cpu().numpy(), LUo)
    assert info[1] == 38
    assert lu_residual(Z, b.a(1).cpu().numpy(), b.piv(1).cpu().numpy()) <= 8 * n * EPS64
    assert info[2] == 1
    assert np.array_equal(b.piv(2).cpu().numpy(), np.arange(n))
    assert not b.a(2).cpu().numpy().any()
