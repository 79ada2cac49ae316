"""Forward error of solves and factorisations against the same operations in
long double: the products that go off an entry are summed apart from it, so
that the result carries a few roundings at its own size and not one for each
product.

The matrices are A = uniform + n I with the equations in a random order: the
products are O(1/n) of the entries they go off, and the conditioning adds
nothing, so the error is the entries' own roundings."""
import numpy as np
import pytest
import torch

import tmv_amd
from checks import EPS64, EPS32

pytestmark = pytest.mark.gpu
WIDE = {False: np.longdouble, True: np.clongdouble}


def wide(a):
    a = np.asarray(a)
    return a.astype(WIDE[np.iscomplexobj(a)])


def matrix(g, n, cplx=False):
    A = g.uniform(-1, 1, (n, n))
    if cplx:
        A = A + 1j * g.uniform(-1, 1, (n, n))
    return (A + n * np.eye(n))[g.permutation(n)]


def host_lu(A):
    """Packed factors and 0-based interchanges of LAPACK's LU."""
    lu, piv = torch.linalg.lu_factor(torch.from_numpy(A))
    return lu.numpy(), piv.numpy().astype(np.int64) - 1


def solve(LU, P, B, trans):
    """A X = B or A^T X = B with given factors, in long double."""
    LU, x, n = wide(LU), wide(B).copy(), len(P)
    swaps = [(k, int(p)) for k, p in enumerate(P) if p != k]
    if not trans:
        for k, p in swaps:
            x[[k, p]] = x[[p, k]]
        for k in range(n):
            x[k + 1:] -= np.outer(LU[k + 1:, k], x[k])
        for k in range(n - 1, -1, -1):
            x[k] /= LU[k, k]
            x[:k] -= np.outer(LU[:k, k], x[k])
    else:
        for k in range(n):
            x[k] /= LU[k, k]
            x[k + 1:] -= np.outer(LU[k, k + 1:], x[k])
        for k in range(n - 1, -1, -1):
            x[:k] -= np.outer(LU[k, :k], x[k])
        for k, p in reversed(swaps):
            x[[k, p]] = x[[p, k]]
    return x


def rms_error(x, ref):
    d = np.abs(wide(x) - ref) ** 2
    return float(np.sqrt(d.mean() / (np.abs(ref) ** 2).mean()))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [33, 64, 200, 256])
def test_batched_transposed_solve(dev, dtype, n):
    """A^T X = B by the workgroup form and the adjoint's.  An entry takes one
    subtraction and one division in U^T and one subtraction in L^T, each of
    at most eps / 2 and rms eps / 2 / sqrt(3): 0.5 eps in all; bar 0.75 eps."""
    eps = EPS64 if dtype == torch.float64 else EPS32
    npt = np.float64 if dtype == torch.float64 else np.float32
    g = np.random.default_rng(n)
    cnt, nr = 8, 2
    b = tmv_amd.Batch([n] * cnt, [nr] * cnt, dtype=dtype)
    w = tmv_amd.Batch([n] * cnt, [nr] * cnt, dtype=dtype)
    grad = tmv_amd.Batch([n] * cnt, [nr] * cnt, dtype=dtype)
    ref = np.empty((cnt, n, nr), np.longdouble)
    for i in range(cnt):
        LU, P = host_lu(matrix(g, n).astype(npt))
        B = g.standard_normal((n, nr)).astype(npt)
        b.a(i).copy_(torch.from_numpy(LU))
        b.piv(i).copy_(torch.from_numpy(P))
        w.b(i).copy_(torch.from_numpy(B))
        ref[i] = solve(LU, P, B, True)
    b.B.copy_(w.B)
    print(f"getrs_batched trans n {n} {dtype}", flush=True)
    tmv_amd.getrs_batched(b, trans=True)
    x = np.stack([b.b(i).cpu().numpy() for i in range(cnt)])
    assert rms_error(x, ref) <= 0.75 * eps
    tmv_amd.gesv_adjoint_batched(b, w, w, grad, grad)
    x = np.stack([grad.b(i).cpu().numpy() for i in range(cnt)])
    assert rms_error(x, ref) <= 0.75 * eps


def factor(A, P):
    """Packed LU of A with given interchanges, in long double."""
    A, n = wide(A).copy(), len(P)
    for k, p in enumerate(P):
        if p != k:
            A[[k, int(p)]] = A[[int(p), k]]
        A[k + 1:, k] /= A[k, k]
        A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
    return A


@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("n", [200, 400])
def test_complex_lu(dev, dtype, n):
    """Complex factors.  An entry takes a rounding at its size for each panel
    of 16 columns before it (25 at n = 400), the rest of its products being
    summed first, and one for each column of its own panel before it (7 on
    average); eps / 2 / sqrt(3) rms each, of the entries that carry most of the
    norm (the diagonal, whose size hides half of that): bar 1.5 eps."""
    npt = np.complex128 if dtype == torch.complex128 else np.complex64
    eps = EPS64 if dtype == torch.complex128 else EPS32
    A = matrix(np.random.default_rng(n), n, cplx=True).astype(npt)
    print(f"getrf_complex n {n} {dtype}", flush=True)
    a = tmv_amd.colmajor(torch.from_numpy(A).cuda())
    piv, info = tmv_amd.getrf_complex(a)
    assert info == 0
    assert rms_error(a.cpu().numpy(), factor(A, piv.cpu().numpy())) <= 1.5 * eps


@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("trans", [False, True])
def test_complex_solve(dev, dtype, trans):
    """Complex solves with given factors.  A sweep goes over an entry once for
    each block of 16 rows before it and sums the products of its own block, so
    an entry of the first sweep takes n / 16 roundings at most and n / 32 on
    average, the second as many: 25 at n = 400, of eps / 2 / sqrt(3) rms a
    component or 1.5 eps; the quotients' own 2 eps beside: bar 3 eps."""
    npt = np.complex128 if dtype == torch.complex128 else np.complex64
    eps = EPS64 if dtype == torch.complex128 else EPS32
    n, g = 400, np.random.default_rng(7)
    LU, P = host_lu(matrix(g, n, cplx=True).astype(npt))
    B = (g.standard_normal((n, 3)) + 1j * g.standard_normal((n, 3))).astype(npt)
    print(f"getrs_complex trans {trans} {dtype}", flush=True)
    lu = tmv_amd.colmajor(torch.from_numpy(LU).cuda())
    x = tmv_amd.colmajor(torch.from_numpy(B).cuda())
    tmv_amd.getrs_complex(lu, torch.from_numpy(P).cuda(), x, trans=trans)
    assert rms_error(x.cpu().numpy(), solve(LU, P, B, trans)) <= 3 * eps
