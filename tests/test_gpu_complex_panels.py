"""Complex LU and solves at the edges of the register panels (16 and 8
columns, one to four rows per thread, above 2048 rows the workgroup panel
first) and of the in-LDS solve (n <= 4096).

Bar: pivots equal to the oracle's where the pivot gap exceeds 64 n eps, ||P A -
L U|| <= 8 n eps ||A||, backward error of both solves <= 8 n eps."""
import numpy as np
import pytest
import torch

import tmv_amd
from checks import EPS64, EPS32
from tmv_amd import rng

pytestmark = pytest.mark.gpu
SEED = 0x7A15EED


def cplx(seed, m, n):
    return rng.uniform_matrix(seed, m, n) + 1j * rng.uniform_matrix(seed + 1, m, n)


def residuals(A, LU, P):
    n = len(A)
    PA = A.copy()
    for i, p in enumerate(P):
        if p != i:
            PA[[i, p]] = PA[[p, i]]
    return np.abs(PA - (np.tril(LU, -1) + np.eye(n)) @ np.triu(LU)).max() / np.abs(A).max()


@pytest.mark.parametrize("dtype,n", [
    (torch.complex128, 15), (torch.complex128, 16), (torch.complex128, 17),
    (torch.complex128, 512), (torch.complex128, 513), (torch.complex128, 1025),
    (torch.complex128, 1037), (torch.complex128, 2048), (torch.complex128, 2049),
    (torch.complex64, 31), (torch.complex64, 530), (torch.complex64, 1100)])
def test_complex_lu_and_solves(orc, dev, dtype, n):
    print(f"complex LU {dtype} {n}", flush=True)
    eps = EPS64 if dtype == torch.complex128 else EPS32
    A = cplx(SEED + 5 * n, n, n)
    B = cplx(SEED + 5 * n + 3, n, 3)
    if dtype == torch.complex64:
        A, B = A.astype(np.complex64).astype(np.complex128), B.astype(np.complex64).astype(np.complex128)
    LU = tmv_amd.colmajor(torch.from_numpy(A).to(dtype).cuda())
    piv, info = tmv_amd.getrf_complex(LU)
    P, lu = piv.cpu().numpy(), LU.cpu().numpy().astype(np.complex128)
    assert info == 0
    if n <= 600:
        _, Po, gaps = orc.getrf_complex(A, gaps=True)
        ok = gaps > 64 * n * eps
        k0 = n if ok.all() else int(np.argmin(ok))
        assert np.array_equal(P[:k0], Po[:k0])
    assert residuals(A, lu, P) <= 8 * n * eps
    for trans in (False, True):
        M = A.T if trans else A
        X = tmv_amd.colmajor(torch.from_numpy(B).to(dtype).cuda())
        tmv_amd.getrs_complex(LU, piv, X, trans=trans)
        x = X.cpu().numpy().astype(np.complex128)
        r = np.abs(B - M @ x).max(axis=0)
        den = np.abs(M).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(B).max(axis=0)
        assert (r <= 8 * n * eps * den).all(), (trans, (r / den).max())


def test_complex_zero_columns_in_panels(dev):
    n = 700
    A = cplx(SEED + 77, n, n)
    A[:, 40] = 0
    A[:, 650] = 0
    LU = tmv_amd.colmajor(torch.from_numpy(A).cuda())
    piv, info = tmv_amd.getrf_complex(LU)
    assert info == 41
    P = piv.cpu().numpy()
    assert P[40] == 40
    assert residuals(A, LU.cpu().numpy(), P) <= 8 * n * EPS64
