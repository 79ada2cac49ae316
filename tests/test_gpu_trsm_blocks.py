"""Solves with many right-hand sides: blocks of 128 rows in groups of 8 steps.

Orders at the edges of a group, of a lane half and of a block, both transposes
(lower and upper, unit and not).  Bar: the backward error of a substitution with
stored factors, 8 n eps.
"""
import pytest
import torch

import tmv_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 127, 128, 129, 200, 261])
@pytest.mark.parametrize("trans", [False, True])
def test_getrs_many_rhs(dt, n, trans):
    nrhs = 18
    gen = torch.Generator().manual_seed(n)
    a = torch.rand(n, n, dtype=dt, generator=gen) * 2 - 1 + n * torch.eye(n, dtype=dt)
    a = a[torch.randperm(n, generator=gen)]
    b = torch.rand(n, nrhs, dtype=dt, generator=gen) * 2 - 1
    lu = tmv_amd.colmajor(a.cuda())
    piv, info = tmv_amd.getrf(lu)
    x = tmv_amd.empty_colmajor(n, nrhs, dt)
    x.copy_(b)
    out = tmv_amd.getrs(lu, piv, x, trans=trans)
    x = (x if out is None else out).cpu().double()
    op = (a.t() if trans else a).double()
    r = (op @ x - b.double()).abs()
    bar = 8 * n * torch.finfo(dt).eps * (op.abs() @ x.abs() + b.double().abs())
    assert bool((r <= bar).all())
