"""GPU test of the moving body's classification where its box is large: boxes
at the size where the kernel changes its form, against the FP64 oracle, and a
box of 2^27 cells (a speed clamp that reaches across the grid), whose classes,
forces and pose equal those of the same body in a box of its own size."""
import numpy as np
import pytest

import oracle_runner
import pylbm
from pylbm import scenarios as sc

pytestmark = pytest.mark.gpu


# the box is the grid where its edge, 2 (ceil(rc) + 3) + 2 + ceil(v_max) + 1,
# exceeds it: 24000 cells, the last small box; 24960, 27000 and more, large ones
@pytest.mark.parametrize("q,grid,shape,v_max", [
    (19, (30, 32, 25), {"kind": 0, "a": 6.2}, 9.0), (27, (30, 32, 26), {"kind": 0, "a": 6.2}, 9.0),
    (27, (40, 40, 40), {"kind": 0, "a": 8.2}, 3.0),
    (19, (40, 48, 33), {"kind": 1, "a": 11.0, "b": 11.0, "c": 17.0}, 20.0),
    (27, (48, 44, 48), {"kind": 2, "a": 12.0, "b": 7.0, "c": 4.0, "r": 1.5}, 9.0)])
def test_classes_and_body_match_the_oracle(q, grid, shape, v_max):
    desc, mac = sc.random_field(*grid, q=q, seed=7, amp=0.02)
    desc = dict(desc, omega=1.25)
    s = np.sin(0.35) / np.sqrt(3.0)
    rigid = {"shape": shape, "x": [grid[0] - 3.3, grid[1] / 2 + 0.2, grid[2] / 2 - 0.4],
             "q": [float(np.cos(0.35)), s, s, s], "v": [0.07, -0.05, 0.06], "omega": [0.004, 0.006, -0.003],
             "density": 2.0, "vMax": v_max, "window": [1, 1, 1], "anchor": [4, 5, 6], "noFluidForce": True}
    with pylbm.Solve(desc) as g:
        g.upload_macro(mac)
        g.attach_rigid(rigid)
        g.step(16)
        cls, st = g.read_classes(), g.read_rigid()
    r = oracle_runner.run(desc, mac, steps=16, want=("body", "cls"), rigid=rigid)
    assert np.array_equal(cls, r["cls"])
    assert np.abs(np.array(st["x"]) - r["body"][-1, :3]).max() < 1e-9


def test_box_of_2_to_the_27_cells():
    n = 512
    desc = {"q": 19, "nx": n, "ny": n, "nz": n, "omega": 1.0 / 0.8, "storage": "f16"}
    mac = np.zeros((n ** 3, 4), np.float32)
    mac[:, 0] = 1.0
    out = []
    for v_max in (600.0, 0.2):
        print("case box 512^3 v_max %g" % v_max, flush=True)
        with pylbm.Solve(desc) as s:
            s.upload_macro(mac)
            s.attach_rigid({"shape": {"kind": 0, "a": 6.3}, "x": [500.4, 500.9, 500.2], "v": [0.06, 0.05, 0.04],
                            "density": 50.0, "vMax": v_max, "window": [1, 1, 1]})
            s.step(3)
            out.append((s.read_classes(), s.read_forces(), s.read_rigid()))
    a, b = out
    assert np.array_equal(a[0], b[0]) and int((a[0] & 1).sum()) > 900
    assert a[2]["x"] == b[2]["x"]
    # the force box does not depend on the clamp
    assert np.array_equal(a[1], b[1]) and np.abs(a[1]).max() > 0
