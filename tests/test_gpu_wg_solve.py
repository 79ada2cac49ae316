"""Batched solves with stored factors, both forms (a workgroup per system up
to 1024 systems, a wave per system above), at the edges of the 16-row
blocks, the wave / workgroup split (n = 64), the 16-column passes and the
largest order, against the oracle's solution of the same factors.

Bar: backward error of every column <= 8 n eps for A X = B and A^T X = B."""
import numpy as np
import pytest
import torch

import tmv_amd
from checks import EPS64, EPS32, backward_error
from tmv_amd import rng

pytestmark = pytest.mark.gpu
SEED = 0x7A15EED


@pytest.mark.parametrize("dtype,count", [(torch.float64, 17), (torch.float64, 1025),
                                         (torch.float32, 17), (torch.float32, 1024)])
def test_stored_factor_solves(orc, dev, dtype, count):
    eps = EPS64 if dtype == torch.float64 else EPS32
    edge = [1, 2, 15, 16, 17, 48, 63, 64, 65, 80, 127, 128, 129, 160, 255, 256, 33]
    ns = (edge + [5] * count)[:count]
    nr = ([1, 2, 3, 16, 17, 4, 1, 33, 1, 2, 0, 5, 1, 2, 3, 17, 1] + [1] * count)[:count]
    b = tmv_amd.Batch(ns, nr, dtype=dtype)
    mats, rhs = {}, {}
    for i in range(len(edge)):
        n, r = ns[i], nr[i]
        A = rng.uniform_matrix(SEED + 31 * i, n, n) + (0.5 * np.eye(n) if n < 4 else 0)
        B = rng.uniform_matrix(SEED + 31 * i + 7, n, max(r, 1))[:, :r]
        if dtype == torch.float32:
            A, B = (M.astype(np.float32).astype(np.float64) for M in (A, B))
        mats[i], rhs[i] = A, B
        b.a(i).copy_(torch.from_numpy(A).to(dtype))
    for i in range(len(edge), count):
        b.a(i).copy_(torch.eye(5, dtype=dtype, device="cuda"))
    tmv_amd.getrf_batched(b)
    for trans in (False, True):
        print(f"getrs {dtype} count {count} trans {trans}", flush=True)
        for i, B in rhs.items():
            b.b(i).copy_(torch.from_numpy(np.ascontiguousarray(B)).to(dtype))
        tmv_amd.getrs_batched(b, trans=trans)
        for i, A in mats.items():
            X = b.b(i).cpu().numpy()
            for c in range(nr[i]):
                be = backward_error(A.T if trans else A, X[:, c], rhs[i][:, c])
                assert be <= 8 * max(ns[i], 4) * eps, (ns[i], c, be)
