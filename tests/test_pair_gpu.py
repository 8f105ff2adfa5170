"""GPU test of the two-step launches (dense_pair.hip): a run in pairs equals the
one-step kernel's bit for bit (populations, macroscopic field, force records),
at the grids where the column cut can go wrong: rows and columns that do not
divide the grid, planes that are not whole layout blocks, one row or one plane,
bodies and walls on the cuts, odd step counts and graph chunks.

set_tile pins a solve to one-step launches, which is what the pairs are
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

STEPS = (4, 2, 17, 1, 40, 3)  # pairs alone, an odd step first, graph chunks


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
    pair, single = run(desc, mac, False), run(desc, mac, True)
    for what, a, b in zip(("mac", "f", "forces"), pair, single):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), what
    assert len(pair[2]) == (sum(STEPS) if desc.get("body") else 0)


@pytest.mark.parametrize("q,grid", [
    (19, (64, 64, 64)), (19, (96, 48, 48)), (19, (128, 70, 37)), (19, (91, 97, 60)), (19, (512, 520, 1)),
    (19, (64, 4, 1100)), (19, (640, 1, 500)), (27, (128, 64, 64)), (27, (100, 83, 61))])
def test_periodic_pairs_equal_single_steps(q, grid):
    desc, mac = sc.random_field(*grid, q=q, seed=sum(grid), amp=0.04)
    check(desc, mac)
    check(dict(desc, force=[1e-5, 2e-6, -1e-6], omegaMinus=1.1), mac)


@pytest.mark.parametrize("q,grid", [(19, (256, 64, 64)), (19, (250, 129, 61)), (27, (192, 72, 72))])
def test_walls_pairs_equal_single_steps(q, grid):
    desc, mac = sc.random_field(*grid, q=q, seed=3, amp=0.03)
    check(dict(desc, walls=[1, 1, 0], wallU=[0.01, -0.02]), mac)
    check(dict(desc, walls=[0, 1, 1], wallU=[-0.01, 0.02], force=[1e-5, 0, 2e-6], omegaMinus=1.2), mac)


@pytest.mark.parametrize("q,grid,body", [
    (19, (256, 128, 64), (11.7, (64.0, 64.5, 32.0))), (19, (230, 121, 61), (9.3, (0.4, 120.2, 30.0))),
    (27, (256, 72, 72), (8.2, (63.5, 36.0, 71.6)))])
@pytest.mark.parametrize("solid_eq", [0, 1])
def test_body_pairs_equal_single_steps(q, grid, body, solid_eq):
    desc, mac = sc.random_field(*grid, q=q, seed=5, amp=0.03)
    check(dict(desc, body={"a": body[0], "centre": list(body[1])}, solidEq=solid_eq, omegaMinus=1.2,
               sponge={"width": 6.0, "axes": [1, 1, 1], "u": [0.03, 0.0, 0.0]}), mac)
