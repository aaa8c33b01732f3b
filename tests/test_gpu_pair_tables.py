"""The point engine's pair terms at every distance: grid points along a line
through one atom, from a hundredth of an Angstrom to beyond the cutoff, against
the oracle.

Two atoms (+1 and -1 e) far apart in a 40 A cubic box (no replication), 4801
points along a spaced 1/120 A: every segment of the real-space tables (r_c / 512
wide) holds a point or two, and so do both sides of the overlap distance (r^2 =
0.1) and the last segment before the cutoff.

Tolerances, from the rounding of one FP32 term (u = 2^-24): r^2 and 1/r are off
by 2 u, the scaled distance r/h (below 512) by 3 u of itself, so the table's
argument by 3 u (alpha r) of x and erfc(x) by at most 2 x^2 + 1 times that ratio,
23 u each at x = 3.3, that is 69 u of a term that has fallen by then to 10^-6 of
those at 1 A: against the condition scale (which adds the Fourier part, 0.3 of
the term at 1 A) below 12 u, and 8 u for the operations, the charge and the FP32
grid: 1.2e-6.  LJ, powers of one reciprocal (1 ulp): 6 (u + 2 u) + 5 u for the
larger power, below 1.6e-6 of each of the two.  FP64: positions of 40 A carry
8e-15 A, so a term of order r^-n at r >= 0.008 A is off by n 1e-12 of itself.
"""
import math

import numpy as np
import pytest

from _parity import say
from conftest import golden  # noqa: F401  (the conftest path set-up)

pytestmark = pytest.mark.gpu

L, N = 40.0, 4801


def _system(pm, r_cut):
    ff = pm.LJForceField("t", {"A": 3.0, "B": 3.0, "P": 3.4}, {"A": 50.0, "B": 50.0, "P": 120.0}, r_cut)
    box = pm.Box(L, L, L, math.pi / 2, math.pi / 2, math.pi / 2)
    x = pm.Crystal("pair", box, ["A", "B"], np.array([[0.0, 0.5], [0.0, 0.5], [0.0, 0.5]]), atom_q=[1.0, -1.0])
    r = np.arange(N) * L / (N - 1)
    return ff, x, np.minimum(r, L - r)


@pytest.mark.parametrize("r_cut", [12.8, 12.0, 8.01])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_real_space_term_at_every_distance(pm, orc, precision, r_cut):
    say(f"case: ion grid line of {N} points, r_c {r_cut} ({precision})")
    ff, x, r = _system(pm, r_cut)
    probe = pm.point_charge(1.0)
    g = pm.energy_grid(x, probe, ff, resolution=(N, 1, 1), units="K", verbose=False, precision=precision,
                       electrostatics=True).data.ravel(order="F")
    o = orc.OracleSystem((L, L, L, math.pi / 2, math.pi / 2, math.pi / 2), x.xf.T, [0, 1], x.atom_q, ff.epsilon_table,
                         ff.sigma2_table, r_cut, np.zeros((0, 3)), [], np.zeros((1, 3)), np.array([1.0]),
                         ewald_precision=1e-6)
    want, scale = o.energy_grid((N, 1, 1)), o.energy_grid_scales((N, 1, 1))
    sel = (r > 0.0) & np.isfinite(want)
    tol = 1.2e-6 if precision == "mixed" else 4e-12
    err = np.abs(g[sel] - want[sel]) / scale[sel]
    say(f"   largest error {err.max():.2e} of the term at r = {r[sel][err.argmax()]:.4f} A")
    assert err.max() <= tol


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lj_term_at_every_distance(pm, precision):
    say(f"case: LJ grid line of {N} points ({precision})")
    ff, x, r = _system(pm, 12.8)
    probe = pm.lj_sphere("P")
    g = pm.energy_grid(x, probe, ff, resolution=(N, 1, 1), units="K", verbose=False,
                       precision=precision).data.ravel(order="F")
    over = r * r < 0.1
    np.testing.assert_array_equal(np.isinf(g), over)
    s2, eps = ff.sigma2("A", "P"), ff.epsilon("A", "P")
    # (a point exactly on the cutoff sphere belongs to either side by rounding)
    ok = ~over & (np.abs(r - 12.8) > 1e-9)
    u = (s2 / r[ok] ** 2) ** 3
    inside = r[ok] ** 2 < 12.8 ** 2
    want = np.where(inside, 4.0 * eps * u * (u - 1.0), 0.0)
    scale = 4.0 * eps * u * (u + 1.0)
    err = np.abs(g[ok] - want) / scale
    say(f"   largest error {err.max():.2e} of the terms")
    assert err.max() <= (1.6e-6 if precision == "mixed" else 1e-11)
