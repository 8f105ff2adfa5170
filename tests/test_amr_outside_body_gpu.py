"""GPU test of an AMR solve whose pinned sphere lies outside the grid, so that
no tile of the finest level exists: the solve steps, its force records are
zeros, and its fields are those of the solve without a body."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "oracle"))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from test_amr_oracle import smooth_field  # noqa: E402

pytestmark = pytest.mark.gpu

N = 16
BODY = {"a": 2.6, "centre": [-20.0, 8.1, 7.9]}


def run(desc, upload):
    with pylbm.Amr(desc) as amr:
        if upload:
            upload(amr)
        mac = smooth_field(N, N, N, 21, amp=0.02)
        mac[:, 1] += 0.04
        amr.upload_macro(mac)
        for n in (1, 2, 2):
            amr.step(n)
        return amr.read_macro(), amr.read_f()[0], amr.read_forces() if "body" in desc else None


def empty(amr):
    amr.upload_topology(np.full(amr.nblocks, -1, np.int32), np.full(amr.max_slots, -1, np.int32))


def level_1_only(amr):
    bs = np.full(amr.nblocks, -1, np.int32)
    bs[21] = 0
    amr.upload_topology(bs, np.array([21] + [-1] * (amr.max_slots - 1), np.int32))
    amr.upload_level_topology(2, np.full(amr.level_blocks(2), -1, np.int32), np.full(amr.max_slots, -1, np.int32))


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("levels,manage,upload", [(2, 0, empty), (2, 2, None), (3, 0, level_1_only)])
def test_body_in_no_tile(q, levels, manage, upload):
    desc = {"q": q, "nx": N, "ny": N, "nz": N, "rb": 4, "maxSlots": 8, "omega": 1 / 0.62, "levels": levels,
            "manageEvery": manage}
    mac, f, forces = run(dict(desc, body=BODY), upload)
    mac0, f0, _ = run(desc, upload)
    assert forces.shape == (5, 6) and not forces.any()
    # a level with a body explodes more directions of its ring, none of which
    # the interior reads
    assert np.array_equal(mac, mac0) and np.array_equal(f, f0)
