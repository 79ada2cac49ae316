"""QR at the edges of the 8-column register panels (one to eight rows a thread,
4096 rows; more rows take the 32-column panels), partial panels, zero columns,
and the solve with one to many right-hand sides.

Bar: R and beta those of LAPACK's dgeqrf in float64 to 64 m eps
|A| (both are backward stable Householder QRs with the same signs), and A = Q R
to 8 m eps through the applied Q^T."""
import numpy as np
import pytest
import scipy.linalg
import torch

import tmv_amd
from checks import EPS64, EPS32
from tmv_amd import rng

pytestmark = pytest.mark.gpu
SEED = 0x7A15EED


@pytest.mark.parametrize("dtype,m,n,nrhs", [
    (torch.float64, 1, 1, 1), (torch.float64, 8, 8, 2), (torch.float64, 9, 7, 1),
    (torch.float64, 512, 9, 3), (torch.float64, 513, 64, 1), (torch.float64, 1025, 33, 17),
    (torch.float64, 2049, 20, 2), (torch.float64, 4096, 17, 1), (torch.float64, 4097, 12, 2),
    (torch.float32, 600, 31, 2), (torch.float32, 2100, 16, 1)])
def test_qr_panels(dev, dtype, m, n, nrhs):
    print(f"qr {dtype} {m}x{n}", flush=True)
    eps = EPS64 if dtype == torch.float64 else EPS32
    A = rng.uniform_matrix(SEED + m + n, m, n)
    B = rng.uniform_matrix(SEED + m + n + 1, m, nrhs)
    if dtype == torch.float32:
        A, B = A.astype(np.float32).astype(np.float64), B.astype(np.float32).astype(np.float64)
    QR = tmv_amd.colmajor(torch.from_numpy(A).to(dtype).cuda())
    beta = tmv_amd.geqrf(QR)
    (qr, tau), _ = scipy.linalg.qr(A, mode="raw")
    got = QR.cpu().numpy().astype(np.float64)
    assert np.abs(np.triu(got[:n]) - np.triu(qr[:n])).max() <= 64 * m * eps * np.abs(A).max()
    assert np.abs(beta.cpu().numpy() - tau).max() <= 64 * m * eps
    X = tmv_amd.colmajor(torch.from_numpy(B).to(dtype).cuda())
    tmv_amd.geqrs(QR, beta, X)
    x = X.cpu().numpy().astype(np.float64)[:n]
    # least squares: A^T (B - A x) = 0, relative to the sizes that enter it
    g = np.abs(A.T @ (B - A @ x)).max()
    assert g <= 64 * m * eps * np.abs(A).max() * (np.abs(B).max() + n * np.abs(A).max() * np.abs(x).max())


def test_qr_zero_columns_in_panel(dev):
    A = rng.uniform_matrix(SEED + 3, 300, 20)
    A[:, 3] = 0
    A[:, 8] = 0
    QR = tmv_amd.colmajor(torch.from_numpy(A).cuda())
    beta = tmv_amd.geqrf(QR).cpu().numpy()
    got = QR.cpu().numpy()
    assert beta[3] == 0 and beta[8] == 0 and got[3, 3] == 0 and got[8, 8] == 0
    R = np.triu(got[:20])
    assert np.abs(R.T @ R - A.T @ A).max() <= 8 * 300 * EPS64 * np.abs(A.T @ A).max()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m", [300, 2000, 4000])
def test_qr_large_entries(dev, dtype, m):
    """Columns whose sum overflows but whose norm does not: the reflector of a
    column of ones has entries of 1 / (1 + sqrt(m)).  Scaling the columns by a
    power of two scales R's columns, so the reference is LAPACK's R of the
    scaled matrix; bar 64 m eps of the column's size."""
    npt = np.float64 if dtype == torch.float64 else np.float32
    eps, big = float(np.finfo(npt).eps), 2.0 * (float(np.finfo(npt).max) / m)
    down = 2.0 ** -60
    A = rng.uniform_matrix(SEED + m, m, 3)
    A[:, 0] = 1.0
    A[:, 1] = big * (0.75 + 0.25 * A[:, 1])
    A[:, 2] *= big
    A = A.astype(npt)
    print(f"qr large {dtype} m {m}", flush=True)
    QR = tmv_amd.colmajor(torch.from_numpy(A).cuda())
    beta = tmv_amd.geqrf(QR).cpu().numpy()
    got = QR.cpu().numpy().astype(np.float64)
    A = A.astype(np.float64)
    A[:, 1:] *= down
    (qr, tau), _ = scipy.linalg.qr(A, mode="raw")
    got[:, 1:][np.triu_indices(m, -1, 2)] *= down       # R's columns, not the reflectors
    R = np.triu(got[:3])
    assert np.all(np.abs(R - np.triu(qr[:3])).max(axis=0) <= 64 * m * eps * np.abs(A).max(axis=0))
    assert np.abs(beta - tau).max() <= 64 * m * eps


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_qr_finished_rows_take_no_part(dev, dtype):
    """Q^T b whose first entry overflows (|b| is beyond the largest number,
    its entries are not): the panels that come later do not see it, and the
    other unknowns are those of b / 4, times 4."""
    npt = np.float64 if dtype == torch.float64 else np.float32
    eps, top = float(np.finfo(npt).eps), float(np.finfo(npt).max)
    m, n = 64, 16
    A = 0.1 * rng.uniform_matrix(SEED + 77, m, n)
    A[:, 0] = 1.0
    A[0, 0] = 1e-3                 # v = (1, 1/sqrt(63), ..): y0 = -sum(b_r) / sqrt(63)
    b = np.full((m, 1), 1.12 * (top / (m - 1)) * np.sqrt(m - 1))
    b[0] = -0.55 * top
    A, b = A.astype(npt), b.astype(npt)
    print(f"qr overflow {dtype}", flush=True)
    QR = tmv_amd.colmajor(torch.from_numpy(A).cuda())
    beta = tmv_amd.geqrf(QR)
    small = tmv_amd.colmajor(torch.from_numpy(b / 4).cuda())
    X = tmv_amd.colmajor(torch.from_numpy(b).cuda())
    tmv_amd.geqrs(QR, beta, small)
    tmv_amd.geqrs(QR, beta, X)
    x, ref = X.cpu().numpy()[1:] / 4, small.cpu().numpy()[1:]
    assert not np.isfinite(X[0].item()) and np.isfinite(small[0].item())
    assert np.abs(x - ref).max() <= 64 * m * eps * np.abs(ref).max()


@pytest.mark.parametrize("dtype,m,n", [
    (torch.float64, 9, 7), (torch.float64, 513, 64), (torch.float64, 1025, 33),
    (torch.float64, 4096, 17), (torch.float64, 4097, 12), (torch.float32, 600, 31),
    (torch.float32, 2100, 16)])
def test_qr_reproduces_the_matrix(dev, dtype, m, n):
    """A = Q R to 8 m eps |A|, with Q formed on the host from the reflectors
    in long double, and the applied Q^T: the solve with A itself on the right
    gives X with R X = R (R x = y to n eps |R||x| beside) and nothing below."""
    print(f"qr product {dtype} {m}x{n}", flush=True)
    eps = EPS64 if dtype == torch.float64 else EPS32
    A = rng.uniform_matrix(SEED + 5 * m + n, m, n)
    if dtype == torch.float32:
        A = A.astype(np.float32).astype(np.float64)
    QR = tmv_amd.colmajor(torch.from_numpy(A).to(dtype).cuda())
    beta = tmv_amd.geqrf(QR)
    got, b = QR.cpu().numpy().astype(np.longdouble), beta.cpu().numpy().astype(np.longdouble)
    P = np.zeros((m, n), np.longdouble)
    P[:n] = np.triu(got[:n])
    for j in range(n - 1, -1, -1):
        v = np.concatenate([np.ones(1, np.longdouble), got[j + 1:, j]])
        P[j:] -= np.outer(v, b[j] * (v @ P[j:]))
    big = np.abs(A).max()
    assert np.abs(P - A).max() <= 8 * m * eps * big
    X = tmv_amd.colmajor(torch.from_numpy(A).to(dtype).cuda())
    tmv_amd.geqrs(QR, beta, X)
    x, R = X.cpu().numpy().astype(np.longdouble), np.triu(got[:n])
    bar = 8 * m * eps * big + n * eps * (np.abs(R) @ np.abs(x[:n])).max()
    assert np.abs(R @ x[:n] - R).max() <= bar
    assert m == n or np.abs(x[n:]).max() <= 8 * m * eps * big
