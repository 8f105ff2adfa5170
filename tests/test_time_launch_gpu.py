"""GPU test of the kernel timing hook: it times the launch that step() takes,
and leaves the solve as it was."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from pylbm import scenarios as sc  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q,grid,storage,body,steps", [
    (19, (256, 128, 128), "f32", (12.0, (64.0, 64.0, 64.0)), 2), (27, (160, 128, 128), "f32", None, 2),
    (9, (960, 480, 1), "f32", (30.0, (240.0, 240.0, 0.0)), 4), (9, (300, 300, 1), "f16", None, 8),
    (19, (256, 128, 128), "f16", None, 1)])
def test_it_times_the_launch_of_a_step(q, grid, storage, body, steps):
    desc, mac = sc.random_field(*grid, q=q, seed=4, amp=0.02)
    desc = dict(desc, storage=storage)
    if body:
        desc["body"] = {"a": body[0], "centre": list(body[1])}
    with pylbm.Solve(desc) as s:
        s.upload_macro(mac)
        s.step(64)
        per_step = min(s.step_timed(128) / 128 for _ in range(3))
        f, records = s.read_f(), s.read_forces(8)
        per_launch = min(s.time_step_kernel(30) for _ in range(3))
        assert np.array_equal(s.read_f(), f) and np.array_equal(s.read_forces(8), records)
        if body:
            n = len(s.read_forces())
            s.step(11)
            assert len(s.read_forces()) == n + 11
        print("ms a step %.5f, a launch %.5f" % (per_step, per_launch), flush=True)
        assert s.launch_steps() == steps
        # gaps between launches, the record's block: a tenth either way, twice
        # that for the box's clock
        assert 0.7 * steps * per_step < per_launch < 1.3 * steps * per_step
