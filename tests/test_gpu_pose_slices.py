"""More poses than one launch takes (2^32 work-items, 2^24 poses of a workgroup
each): every pose of a call of 2^24 + 5 gets its own result.  The poses repeat a
few distinct ones, whose results from a small call must come back bit for bit.
"""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu

N = (1 << 24) + 5
DISTINCT = 61  # odd: slices of the call start at different ones


def test_calls_of_more_poses_than_a_launch(pm):
    say(f"case: {N} one-site poses in one atom, energies and forces")
    ff = pm.LJForceField("t", {"A": 3.0, "P": 3.2}, {"A": 50.0, "P": 90.0}, 6.0)
    box = pm.Box(13.0, 13.0, 13.0, math.pi / 2, math.pi / 2, math.pi / 2)
    x = pm.Crystal("one", box, ["A"], np.array([[0.5], [0.4], [0.3]]))
    few = np.random.default_rng(3).random((DISTINCT, 1, 3))
    many = few[np.arange(N) % DISTINCT]
    want = pm.vdw_energies(x, ["P"], few, ff)
    assert len(set(want)) > 10  # (poses beyond the cutoff are all zero)
    got = pm.vdw_energies(x, ["P"], many, ff)
    assert np.array_equal(got, want[np.arange(N) % DISTINCT])
    say("   energies of every pose")
    fw = pm.device.framework(x, ff)
    e, g = pm.device.pose_gradients(fw, ff, None, [ff.index("P")], [0.0], few, "fp64")
    em, gm = pm.device.pose_gradients(fw, ff, None, [ff.index("P")], [0.0], many, "fp64")
    assert np.array_equal(em, e[np.arange(N) % DISTINCT]) and np.array_equal(gm, g[np.arange(N) % DISTINCT])
