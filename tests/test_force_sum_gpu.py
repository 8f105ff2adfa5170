"""GPU test of the force records of large bodies, whose boundary cells are
summed in chunks by several blocks: against the FP64 oracle, the same bits from
every launch form and from the serve loop, and without a launch waiting for the
sum."""
import os
import sys

import numpy as np
import pytest

import oracle_runner

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from pylbm import scenarios as sc  # noqa: E402

pytestmark = pytest.mark.gpu


def solve(q, grid, radius, centre, storage="f32"):
    desc, mac = sc.random_field(*grid, q=q, seed=9, amp=0.02)
    return dict(desc, storage=storage, omegaMinus=1.2, omega=1.5, body={"a": radius, "centre": list(centre)}), mac


# one chunk of 1024 boundary cells, two, five, ten (more than a wave of chunk
# sums is below); 2D across the periodic edge
@pytest.mark.parametrize("q,grid,radius,centre", [
    (19, (32, 32, 32), 6.2, (16.0, 15.6, 16.3)), (19, (40, 40, 40), 9.4, (20.0, 19.7, 20.2)),
    (27, (48, 48, 48), 15.3, (24.0, 24.4, 23.6)), (19, (64, 64, 64), 23.8, (32.2, 32.0, 31.7)),
    (9, (1200, 900, 1), 401.0, (3.0, 450.0, 0.0))])
def test_records_match_the_oracle(q, grid, radius, centre):
    desc, mac = solve(q, grid, radius, centre)
    with pylbm.Solve(desc) as s:
        s.upload_macro(mac)
        s.step(5)
        f = s.read_forces()
    r = oracle_runner.run(desc, mac, steps=5, threads=4, want=("force",))["force"]
    scale = np.abs(r[:, :3]).max()
    assert f.shape == (5, 6)
    # fp32 populations: 2^-24 of each link's momentum, 2 w, over the cells' links
    assert np.abs(f[:, :3] - r[:, :3]).max() < 1e-5 * scale + 1e-6 * radius
    assert np.abs(f[:, 3:] - r[:, 3:]).max() < 1e-5 * scale * radius + 1e-6 * radius * radius


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("q,grid,radius", [(19, (96, 80, 80), 33.0), (27, (112, 110, 110), 52.0), (9, (700, 500, 1), 230.0)])
def test_every_form_gives_the_same_records(q, grid, radius, storage):
    desc, mac = solve(q, grid, radius, [n / 2.0 + 0.3 for n in grid], storage)
    out = []
    forms = (1, 2) if q == 9 or storage == "f32" else (1,)
    for n in forms + ((0,) if q == 9 else ()):
        with pylbm.Solve(desc) as s:
            s.set_launch_steps(n)
            s.upload_macro(mac)
            for k in (3, 1, 20, 40):
                s.step(k)
            out.append((s.read_forces(), s.read_macro()))
    with pylbm.Server(budget_bytes=2e9, chunk_steps=16) as sv:
        # two residents of one class, summed in the same launches
        tickets = [sv.submit(desc, mac, 64) for _ in range(2)]
        for t in tickets:
            sv.wait(t)
            out.append((sv.read_forces(t, 64), sv.read_macro(t)))
            sv.release(t)
    assert out[0][0].shape == (64, 6)
    for f, m in out[1:]:
        assert np.array_equal(f, out[0][0]) and np.array_equal(m, out[0][1])


@pytest.mark.parametrize("q,n,storage", [(19, 120, "f32"), (19, 96, "f16")])
def test_a_step_does_not_wait_for_the_sum(q, n, storage):
    best = {}
    for radius in (6.0, n / 4.0):
        desc, mac = solve(q, (n, n, n), radius, (n / 2.0, n / 2.0, n / 2.0), storage)
        with pylbm.Solve(desc) as s:
            s.set_launch_steps(1)
            s.upload_macro(mac)
            s.step(40)
            best[radius] = min(s.step_timed(66) / 66 for _ in range(8))
    print("ms a step", best, flush=True)
    # with one block summing 1.65 and 1.5 times; a body's own cells cost a quarter
    # at most
    assert best[n / 4.0] < 1.37 * best[6.0]
