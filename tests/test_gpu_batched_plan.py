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
