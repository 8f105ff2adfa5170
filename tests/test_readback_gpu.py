"""GPU test of the copies back to the host: a field large enough to come in
chunks by several threads, of a size that no chunk divides, alone and from two
threads at once, and the force ring read across its end."""
import os
import sys
import threading

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "getting-air_amd"))

import pylbm  # noqa: E402
from pylbm import scenarios as sc  # noqa: E402

pytestmark = pytest.mark.gpu


def test_large_fields_come_back_whole():
    fields = [sc.random_field(2101, 1009, 1, q=9, seed=k, amp=0.03) for k in (1, 2)]  # 33.9 MB each
    with pylbm.Solve(fields[0][0]) as a, pylbm.Solve(fields[1][0]) as b:
        solves = (a, b)
        for s, (_, mac) in zip(solves, fields):
            s.upload_macro(mac)
            assert np.array_equal(s.read_macro(), mac)
        got = [None, None]

        def read(k):
            got[k] = [solves[k].read_macro() for _ in range(3)]

        threads = [threading.Thread(target=read, args=(k,)) for k in (0, 1)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for k in (0, 1):
            assert all(np.array_equal(m, fields[k][1]) for m in got[k])


def test_force_records_across_the_ring():
    desc, mac = sc.random_field(16, 16, 1, q=9, seed=3, amp=0.03)
    with pylbm.Solve(dict(desc, body={"a": 2.5, "centre": [8.0, 8.0, 0.0]})) as s:
        s.upload_macro(mac)
        s.step((1 << 16) - 30)
        head = s.read_forces(20)
        s.step(50)
        tail = s.read_forces(50)  # the last 20 of them past the ring's end
        assert len(head) == 20 and len(tail) == 50
        assert np.array_equal(s.read_forces(70)[:20], head)
        assert np.array_equal(s.read_forces(70)[20:], tail)
        assert len(s.read_forces()) == 1 << 16
        assert np.array_equal(s.read_forces()[-70:-50], head)
        assert np.array_equal(s.read_forces(20), tail[-20:])
        assert s.read_forces(0).shape == (0, 6)
