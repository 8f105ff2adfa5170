"""GPU test of calls that advance a 2D solve by fewer steps than a launch
holds, a page that draws every frame: mixed with whole launches they equal
one-step launches bit for bit on both sides of the rule's lines, and on the
grids where a shorter launch would be the slower form they take no longer than
one-step launches."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from pylbm import scenarios as sc  # noqa: E402

pytestmark = pytest.mark.gpu

CALLS = (1, 1, 2, 1, 8, 3, 2, 2, 9, 10, 1, 70, 6, 2, 5)


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("grid", [(48, 40), (300, 200), (700, 300), (2048, 2047), (2048, 2048), (2500, 1700)])
@pytest.mark.parametrize("body", [False, True])
def test_short_advances_equal_single_steps(grid, storage, body):
    desc, mac = sc.random_field(*grid, 1, q=9, seed=sum(grid), amp=0.03)
    desc = dict(desc, storage=storage, walls=[0, 1, 0], wallU=[0.01, -0.02])
    if body:
        desc["body"] = {"a": min(grid) / 5.0, "centre": [grid[0] / 3.0, grid[1] / 2.0, 0.0]}
    out = []
    for steps in (0, 1):
        with pylbm.Solve(desc) as s:
            s.set_launch_steps(steps)
            s.upload_macro(mac)
            fields = []
            for n in CALLS:
                s.step(n)
                fields.append(s.read_macro() if grid[0] < 1000 else None)
            out.append((fields, s.read_macro(), s.read_f(), s.read_forces() if body else None))
    several, single = out
    for a, b in zip(several[0], single[0]):
        assert a is None or np.array_equal(a, b)
    assert np.array_equal(several[1], single[1]) and np.array_equal(several[2], single[2])
    if body:
        assert len(several[3]) == sum(CALLS) and np.array_equal(several[3], single[3])


# a shorter launch takes 1.4, 1.7 and 1.2 times as long
@pytest.mark.parametrize("storage,n,most", [("f32", 1, 1.2), ("f16", 1, 1.2), ("f16", 2, 1.1)])
def test_short_advances_take_no_longer_than_single_steps(storage, n, most):
    desc, mac = sc.random_field(4096, 2048, 1, q=9, seed=1, amp=0.01)
    best = [1e9, 1e9]
    with pylbm.Solve(dict(desc, storage=storage)) as a, pylbm.Solve(dict(desc, storage=storage)) as b:
        b.set_launch_steps(1)
        for s in (a, b):
            s.upload_macro(mac)
        for _ in range(40):
            for k, s in enumerate((a, b)):
                best[k] = min(best[k], s.step_timed(n))
    print("ms", best, flush=True)
    assert best[0] < most * best[1]
