"""GPU test of the launch forms: each is forced and asserted, on grids small
enough to run every instantiation of the two-step kernel (lattice, general,
body force, planes of whole layout blocks or not) and every step count of a 2D
launch, and equals one-step launches bit for bit (populations, macroscopic
field, force records).  The engine's own choice is pinned on grids of each
kind."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from pylbm import scenarios as sc  # noqa: E402

pytestmark = pytest.mark.gpu

STEPS = (4, 2, 17, 1, 40, 3)  # whole launches, an odd step first, graph chunks
FORCE = {"force": [1e-5, 2e-6, -1e-6], "omegaMinus": 1.1}


def run(desc, mac, steps):
    with pylbm.Solve(desc) as s:
        s.set_launch_steps(steps)
        assert s.launch_steps() == steps
        s.upload_macro(mac)
        for n in STEPS:
            s.step(n)
        assert s.launch_steps() == steps
        forces = s.read_forces() if desc.get("body") else np.zeros((0, 6))
        return s.read_macro(), s.read_f(), forces


def check(desc, mac, *counts):
    single = run(desc, mac, 1)
    assert np.isfinite(single[0]).all()
    assert len(single[2]) == (sum(STEPS) if desc.get("body") else 0)
    for n in counts:
        for what, a, b in zip(("mac", "f", "forces"), run(desc, mac, n), single):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (what, n)


# whole layout blocks to a plane, then not: one column and several, columns and
# rows cut short, one row, one plane, fewer cells than a column's row
ALIGNED = [(72, 16, 9), (130, 32, 3), (64, 1, 20), (192, 41, 1), (8, 24, 11)]
RAGGED = [(70, 15, 9), (131, 29, 4), (67, 1, 13), (150, 31, 1), (5, 7, 3)]


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("grid", ALIGNED + RAGGED)
def test_periodic(q, grid):
    assert (grid[0] * grid[1] % 64 == 0) == (grid in ALIGNED)
    desc, mac = sc.random_field(*grid, q=q, seed=sum(grid), amp=0.04)
    check(desc, mac, 2)
    check(dict(desc, **FORCE), mac, 2)


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("grid", ALIGNED + RAGGED)
def test_walls(q, grid):
    desc, mac = sc.random_field(*grid, q=q, seed=3, amp=0.03)
    check(dict(desc, walls=[1, 1, 0], wallU=[0.01, -0.02]), mac, 2)
    check(dict(desc, walls=[1, 1, 1], wallU=[-0.01, 0.02], **FORCE), mac, 2)


# the sphere inside a column; across the columns' and rows' cut (x = 64; rows of
# 11 and 8 or 9); across a periodic corner; on a wall
@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("grid", [(136, 32, 18), (133, 33, 17)])
@pytest.mark.parametrize("body", [(4.3, (30.2, 9.5, 8.0)), (6.1, (64.2, 16.4, 8.3)), (3.2, (0.3, 0.4, 0.2)),
                                  (5.2, (70.0, 20.0, 8.1))])
@pytest.mark.parametrize("solid_eq", [0, 1])
def test_bodies(q, grid, body, solid_eq):
    desc, mac = sc.random_field(*grid, q=q, seed=5, amp=0.03)
    desc = dict(desc, body={"a": body[0], "centre": list(body[1])}, solidEq=solid_eq)
    check(dict(desc, omegaMinus=1.2, sponge={"width": 3.0, "axes": [1, 1, 1], "u": [0.03, 0.0, 0.0]}), mac, 2)
    check(dict(desc, walls=[0, 1, 0], **FORCE), mac, 2)


# grids that the engine's choice sends to pairs
@pytest.mark.parametrize("q,grid,extra", [
    (19, (122, 122, 122), {}), (19, (190, 99, 99), FORCE), (27, (100, 100, 150), {}), (27, (190, 99, 99), FORCE),
    (27, (255, 129, 130), {"walls": [0, 1, 1], "wallU": [0.01, -0.02]}),
    (27, (255, 130, 130), dict(FORCE, walls=[1, 1, 0])), (19, (256, 128, 64), {"walls": [0, 1, 0]})])
def test_chosen_pairs(q, grid, extra):
    desc, mac = sc.random_field(*grid, q=q, seed=11, amp=0.03)
    desc = dict(desc, **extra)
    with pylbm.Solve(desc) as s:
        assert s.launch_steps() == 2
    check(desc, mac, 2)


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("grid,most", [((16, 16), 8), ((65, 17), 8), ((161, 160), 8), ((36, 500), 8), ((400, 390), 4)])
def test_2d_counts(grid, most, storage):
    desc, mac = sc.random_field(*grid, 1, q=9, seed=sum(grid), amp=0.04)
    desc = dict(desc, storage=storage)
    with pylbm.Solve(desc) as s:
        assert s.launch_steps() == most
    check(dict(desc, force=[1e-5, 2e-6, 0.0], walls=[0, 1, 0], wallU=[0.01, -0.02]), mac, *range(2, most + 1))
    check(dict(desc, body={"a": min(grid) / 4.0, "centre": [grid[0] / 3.0, grid[1] / 2.0, 0.0]}, omegaMinus=1.2), mac,
          *range(2, most + 1))


def steps_of(desc, n=0, tile=False):
    with pylbm.Solve(desc) as s:
        if tile:
            t = s.info()
            s.set_tile(t["block_x"], t["block_y"], t["flags"])
            assert s.launch_steps() == 1
        s.set_launch_steps(n)
        return s.launch_steps()


def test_choice_and_refusals():
    d3, _ = sc.random_field(128, 128, 96, q=19, seed=1, amp=0.01)
    small, _ = sc.random_field(32, 16, 16, q=19, seed=1, amp=0.01)
    d2, _ = sc.random_field(200, 200, 1, q=9, seed=1, amp=0.01)
    body = {"a": 4.0, "centre": [16.0, 8.0, 8.0]}
    # the engine's choice, also after a tile has pinned one step
    assert [steps_of(d, 0, t) for d in (d3, small, d2) for t in (False, True)] == [2, 2, 1, 1, 8, 8]
    assert steps_of(dict(d3, storage="f16")) == 1 and steps_of(dict(d3, diffuse=1, body=body)) == 1
    assert steps_of(small, 2) == 2 and steps_of(d2, 5) == 5
    for desc, n, code in ((d3, 3, -4), (d3, -1, -1), (d2, 9, -1), (dict(d3, storage="bf16"), 2, -4),
                          (dict(small, diffuse=1, body=body), 2, -4),
                          (sc.random_field(15, 40, 1, q=9, seed=1, amp=0.01)[0], 2, -4)):
        with pytest.raises(pylbm.LbmError) as e:
            steps_of(desc, n)
        assert e.value.code == code
    desc, mac = sc.random_field(128, 64, 64, q=19, seed=1, amp=0.01)
    with pylbm.Solve(desc) as s:
        s.upload_macro(mac)
        before = s.info()["device_bytes"]
        for n in (1, 2, 0, 1, 0):
            s.set_launch_steps(n)
        assert s.info()["device_bytes"] == before
        s.attach_rigid({"shape": {"kind": 0, "a": 5.2}, "x": [50.0, 30.0, 30.0]})
        assert s.launch_steps() == 1
        with pytest.raises(pylbm.LbmError):
            s.set_launch_steps(2)
