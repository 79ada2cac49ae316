"""Plans of batched solves: what a forced schedule refuses, and that a system's
result does not depend on the batch that it is in."""
import numpy as np
import pytest
import torch

import tmv_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule,cap", [(0, 16), (1, 32), (2, 64)])
def test_forced_schedule_refuses_wide_rhs_per_wave(dev, schedule, cap):
    """A system of n <= min(split, the schedule's cap) with more than 8
    right-hand sides is refused, and the plan stays as it was."""
    plan = tmv_amd.BatchPlan([cap, 100], [9, 16])
    before = plan.describe()
    for split in (cap, 64, 1000):
        with pytest.raises(tmv_amd.TmvxError):
            plan.set(schedule, split, 2)
    assert plan.describe() == before
    plan.set(schedule, cap - 1, 2)
    tmv_amd.BatchPlan([cap, 100], [8, 16]).set(schedule, 64, 2)
    tmv_amd.BatchPlan([cap + 1, 100], [9, 16]).set(schedule, cap, 2)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_result_does_not_depend_on_the_batch(dev, dtype):
    """Bit for bit the same factors, interchanges and solutions by itself, in
    a batch of its like and among others in another order, with orders on both
    sides of 32 and 64."""
    ns = [1, 8, 31, 32, 33, 48, 63, 64, 65, 100, 127, 128]
    nr = [1, 2, 4, 1, 9, 3, 1, 16, 1, 5, 16, 2]
    g = np.random.default_rng(3)
    mats = [torch.from_numpy(g.uniform(-1, 1, (n, n))).to(dtype) for n in ns]
    rhs = [torch.from_numpy(g.uniform(-1, 1, (n, r))).to(dtype) for n, r in zip(ns, nr)]

    def run(which, fill):
        idx = list(which)
        b = tmv_amd.Batch([ns[i] for i in idx] + fill, [nr[i] for i in idx] + [1] * len(fill),
                          dtype=dtype)
        b.A.fill_(1.0)
        for k, i in enumerate(idx):
            b.a(k).copy_(mats[i])
            b.b(k).copy_(rhs[i])
        tmv_amd.gesv_batched(tmv_amd.BatchPlan(b), b)
        return {i: (b.a(k).cpu(), b.piv(k).cpu(), b.b(k).cpu(), b.info[k].item())
                for k, i in enumerate(idx)}

    print(f"batch independence {dtype}", flush=True)
    every = run(range(len(ns)), [])
    among = run(reversed(range(len(ns))), [1 + 7 * i % 128 for i in range(300)])
    for i in range(len(ns)):
        alone = run([i], [])[i]
        for other in (every[i], among[i]):
            assert alone[3] == other[3] == 0
            for u, v in zip(alone[:3], other[:3]):
                assert torch.equal(u, v), ns[i]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 3, 32, 33, 64])
def test_columns_do_not_depend_on_their_number(dev, dtype, n):
    """Right-hand sides go four at a time and a last one by itself: each
    column is bit for bit that of a solve of its own."""
    g = np.random.default_rng(n)
    A = torch.from_numpy(g.uniform(-1, 1, (n, n))).to(dtype)
    B = torch.from_numpy(g.standard_normal((n, 16))).to(dtype)

    def run(counts):
        b = tmv_amd.Batch([n] * len(counts), [len(c) for c in counts], dtype=dtype)
        for k, c in enumerate(counts):
            b.a(k).copy_(A)
            b.b(k).copy_(B[:, c])
        tmv_amd.gesv_batched(tmv_amd.BatchPlan(b), b)
        return [b.b(k).cpu() for k in range(len(counts))]

    print(f"columns n {n} {dtype}", flush=True)
    single = torch.cat(run([[c] for c in range(16)]), dim=1)
    for r, x in zip(range(17), run([list(range(r)) for r in range(17)])):
        assert torch.equal(x, single[:, :r]), r
