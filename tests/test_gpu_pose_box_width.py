"""A box exactly as wide as the cutoff sphere: an atom just less than half a box
away is inside the cutoff, while from coordinates rounded to FP32 its image on the
other side is the nearest; in a skewed box that one is far away.  The pair's energy
and force must be there."""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu


def _pairs(n):
    """Fractions z of an atom and z + 1/2 + 1e-9 of a pose: the nearest image of the
    atom lies 1/2 - 1e-9 above; that of their FP32 values 1/2 below."""
    z = np.random.default_rng(7).uniform(0.01, 0.49, 400)
    t = z + 0.5 + 1e-9
    d = z.astype(np.float32) - t.astype(np.float32)
    keep = (d - np.rint(d) < 0) & (z - t < -0.5)
    return list(zip(z[keep][:n], t[keep][:n]))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_pairs_half_a_box_apart(pm, precision):
    box = pm.Box(26.0, 25.0, 24.0, math.radians(75.0), math.radians(80.0), math.radians(85.0))
    f = box.f_to_c
    assert f[1, 0] == 0.0 and f[2, 0] == 0.0 and f[2, 1] == 0.0
    r_c = 0.5 * f[2, 2] * (1.0 - 1e-12)  # the third axis' width is the smallest
    say(f"case: pairs at half of a box {f[2, 2]:.3f} A wide, cutoff {r_c:.3f} A ({precision})")
    ff = pm.LJForceField("t", {"A": 3.4, "P": 3.6}, {"A": 80.0, "P": 120.0}, r_c)
    pairs = _pairs(8)
    assert len(pairs) == 8
    for z, t in pairs:
        dz = z - t + 1.0
        dy = -f[1, 2] * dz / f[1, 1]
        dx = -(f[0, 1] * dy + f[0, 2] * dz) / f[0, 0]
        x = pm.Crystal("one", box, ["A"], np.array([[0.5], [0.5], [z]]))
        xf = np.array([[[0.5 - dx, 0.5 - dy, t]]])
        r = f[2, 2] * dz
        assert r < r_c
        u = (ff.sigma2("A", "P") / r ** 2) ** 3
        e4 = 4.0 * ff.epsilon("A", "P")
        tol = 1e-10 if precision == "fp64" else 2e-6  # six powers of one FP32 reciprocal
        v = pm.vdw_energies(x, ["P"], xf, ff, precision=precision)
        assert abs(v[0] - e4 * u * (u - 1.0)) <= tol * e4 * u
        fw = pm.device.framework(x, ff)
        g = pm.device.pose_gradients(fw, ff, None, [ff.index("P")], [0.0], xf, precision)[1]
        assert abs(g[0, 0, 2] - 6.0 * e4 * u * (2.0 * u - 1.0) / r) <= tol * 6.0 * e4 * u / r
