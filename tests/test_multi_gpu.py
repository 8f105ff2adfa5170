"""GPU test of the D2Q9 launches of several steps (dense_multi.hip): a run in
such launches equals the one-step kernel's bit for bit (populations, macroscopic
field, force records), at the grids where the tiling can go wrong: the smallest
and largest of each tile's range, tiles cut to a column or a row, frames that
wrap around the grid, grids that are not whole layout blocks, bodies and walls
on the cuts, step counts that leave a short launch, and graph chunks.

set_tile pins a solve to one-step launches, which is what the others are
compared with."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from pylbm import scenarios as sc  # noqa: E402

pytestmark = pytest.mark.gpu

STEPS = (8, 4, 17, 1, 150, 3)  # whole launches, short ones, graph chunks

# Small (16^2 to 400 tiles of 8 x 8), Deep (to 512 of 16 x 16), Wide; narrow
# grids that only the smaller tiles fit
GRIDS = [(16, 16), (64, 64), (65, 17), (160, 160), (161, 160), (24, 900), (353, 351), (384, 352), (50, 5000), (36, 5000),
         (35, 4001),
         (517, 203), (20, 2000), (16, 4000), (15, 40)]


def run(desc, mac, one_step):
    with pylbm.Solve(desc) as s:
        if one_step:
            t = s.info()
            s.set_tile(t["block_x"], t["block_y"], t["flags"])
        s.upload_macro(mac)
        for n in STEPS:
            s.step(n)
        forces = s.read_forces() if desc.get("body") else np.zeros((0, 6))
        return s.read_macro(), s.read_f(), forces


def check(desc, mac):
    several, single = run(desc, mac, False), run(desc, mac, True)
    for what, a, b in zip(("mac", "f", "forces"), several, single):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), what
    assert len(several[2]) == (sum(STEPS) if desc.get("body") else 0)


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_several_steps_equal_single_steps(nx, ny, storage):
    desc, mac = sc.random_field(nx, ny, 1, q=9, seed=nx + ny, amp=0.04)
    desc = dict(desc, storage=storage)
    check(desc, mac)
    check(dict(desc, force=[1e-5, 2e-6, 0.0], walls=[0, 1, 0], wallU=[0.01, -0.02], omegaMinus=1.1), mac)
    check(dict(desc, walls=[1, 1, 0]), mac)
    check(dict(desc, solidEq=1, omegaMinus=1.2, body={"a": min(nx, ny) / 4.0, "centre": [nx / 3.0, ny / 2.0, 0.0]},
               sponge={"width": 6.0, "axes": [1, 1, 0], "u": [0.03, 0.0, 0.0]}), mac)
    check(dict(desc, walls=[0, 1, 0], force=[1e-5, 0.0, 0.0], body={"a": 2.3, "centre": [nx - 0.5, 0.4, 0.0]}), mac)
