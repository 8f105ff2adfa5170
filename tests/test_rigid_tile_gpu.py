"""GPU test of the tile flags under a moving body: a caller's stay through any
number of attachments, the default's are those of the rigid step."""
import pytest

import pylbm
from pylbm import scenarios as sc

pytestmark = pytest.mark.gpu

RIGID = {"shape": {"kind": 0, "a": 5.2}, "x": [50.0, 30.0, 30.0], "v": [0.02, 0.0, 0.0]}


def flags(grid, tile, walls):
    desc, mac = sc.random_field(*grid, q=19, seed=2, amp=0.02)
    with pylbm.Solve(dict(desc, walls=walls)) as s:
        if tile is not None:
            s.set_tile(128, 1, tile)
        s.upload_macro(mac)
        out = []
        for _ in range(3):
            s.attach_rigid(RIGID)
            s.step(2)
            out.append(s.info()["flags"])
        return out


@pytest.mark.parametrize("walls", [[0, 0, 0], [0, 1, 0]])
@pytest.mark.parametrize("tile", [0x4, 0x5, 0x6, 0x47])
def test_a_callers_flags_survive_every_attach(tile, walls):
    assert flags((100, 60, 60), tile, walls) == [tile] * 3


# 55 MB, default launches that stay in the last-level cache; 640 MB, streamed
@pytest.mark.parametrize("grid", [(100, 60, 60), (100, 210, 200)])
def test_the_default_is_non_temporal(grid):
    assert flags(grid, None, [0, 0, 0]) == [0x66] * 3
