"""Batched LU + solve at the edges of its panels (8-column blocks, the 32 /
64-column kernels, the 64-column split of larger systems), with every number
of right-hand sides, exact ties and rows that need interchanges, against the
oracle; bar as in test_gpu_batched."""
import numpy as np
import pytest
import scipy.linalg
import torch

import tmv_amd
from checks import EPS64, EPS32, lu_residual, backward_error
from tmv_amd import rng

pytestmark = pytest.mark.gpu
SEED = 0x7A15EED


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("rot", [0, 5, 11])
def test_batched_edges(orc, dev, dtype, rot):
    eps = EPS64 if dtype == torch.float64 else EPS32
    ns = [1, 7, 8, 9, 24, 25, 31, 32, 33, 40, 41, 63, 64, 65, 66, 72, 79, 80, 81, 96, 112, 113,
          127, 128]
    nrhs = [(i + rot) % 17 for i in range(len(ns))]
    print(f"batched edges {dtype} rot {rot}", flush=True)
    b = tmv_amd.Batch(ns, nrhs, dtype=dtype)
    As, Bs = [], []
    for i, (n, r) in enumerate(zip(ns, nrhs)):
        A = rng.uniform_matrix(SEED + 17 * i + rot, n, n) + (np.eye(n) if n < 4 else 0)
        A = A[::-1].copy()
        B = rng.uniform_matrix(SEED + 17 * i + 9 + rot, n, max(r, 1))[:, :r]
        if dtype == torch.float32:
            A, B = (M.astype(np.float32).astype(np.float64) for M in (A, B))
        As.append(A)
        Bs.append(B)
        b.a(i).copy_(torch.from_numpy(A).to(dtype))
        if r:
            b.b(i).copy_(torch.from_numpy(np.ascontiguousarray(B)).to(dtype))
    tmv_amd.gesv_batched(tmv_amd.BatchPlan(b), b)
    assert not b.info.cpu().numpy().any()
    for i, n in enumerate(ns):
        P = b.piv(i).cpu().numpy()
        _, Po, gaps = orc.getrf(As[i], gaps=True)
        ok = gaps > 64 * n * eps
        k0 = n if ok.all() else int(np.argmin(ok))
        assert np.array_equal(P[:k0], Po[:k0]), n
        assert lu_residual(As[i], b.a(i).cpu().numpy(), P) <= 8 * max(n, 4) * eps, n
        X = b.b(i).cpu().numpy()
        for c in range(nrhs[i]):
            assert backward_error(As[i], X[:, c], Bs[i][:, c]) <= 8 * max(n, 4) * eps, (n, c)


def test_batched_ties(orc, dev):
    mats = [scipy.linalg.hadamard(n).astype(np.float64) for n in (8, 16, 32, 64, 128)]
    b = tmv_amd.Batch([len(H) for H in mats])
    for i, H in enumerate(mats):
        b.a(i).copy_(torch.from_numpy(H))
    tmv_amd.gesv_batched(tmv_amd.BatchPlan(b), b)
    for i, H in enumerate(mats):
        LUo, Po = orc.getrf(H)
        assert np.array_equal(b.piv(i).cpu().numpy(), Po), len(H)
        assert np.array_equal(b.a(i).cpu().numpy(), LUo), len(H)
