"""Batched GEMM with one problem a workgroup and with four (8192 problems up).

Counts around the change and not a multiple of four, sizes at the edges of a 32 x
32 block and of the 16 deep steps.  Bar: k eps |A||B| per entry (the error of a
sum of k products).
"""
import numpy as np
import pytest
import torch

import tmv_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("count", [1, 8191, 8192, 8195])
def test_gemm_batched_groups(dt, count):
    pool = np.array([1, 2, 3, 15, 16, 17, 31, 32, 33, 40])
    ns = pool[np.arange(count) % len(pool)].astype(np.int32)
    gen = torch.Generator().manual_seed(3)
    total = int((ns.astype(np.int64) ** 2).sum())
    av = torch.rand(total, dtype=dt, generator=gen) * 2 - 1
    bv = torch.rand(total, dtype=dt, generator=gen) * 2 - 1
    a = tmv_amd.Batch(ns, dtype=dt, A=av.cuda())
    b = tmv_amd.Batch(ns, dtype=dt, A=bv.cuda())
    c = tmv_amd.Batch(ns, dtype=dt)
    c.A.fill_(float("nan"))
    tmv_amd.gemm_batched(a.d_n, a.d_n, a.d_n, a.pA, b.pA, c.pA, dtype=dt)
    out = c.A.cpu().double()
    off = np.concatenate([[0], np.cumsum(ns.astype(np.int64) ** 2)])
    eps = torch.finfo(dt).eps
    for n in set(int(x) for x in ns):
        ids = np.nonzero(ns == n)[0]
        pick = torch.from_numpy(off[ids][:, None] + np.arange(n * n)[None, :])
        A, B, C = (v[pick].view(-1, n, n).transpose(1, 2).contiguous()
                   for v in (av.double(), bv.double(), out))
        bar = (n + 2) * eps * (A.abs() @ B.abs())
        assert bool(((C - A @ B).abs() <= bar).all()), n


@pytest.mark.parametrize("dt,count", [(torch.float64, 2047), (torch.float64, 2048),
                                      (torch.float64, 2051), (torch.float32, 4095),
                                      (torch.float32, 4096), (torch.float32, 4099)])
def test_gemm_batched_where_groups_begin(dt, count):
    """Four problems a workgroup from 2048 (FP64) or 4096 (FP32) on."""
    test_gemm_batched_groups(dt, count)
