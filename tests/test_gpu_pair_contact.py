"""Grid points exactly on an atom: a point charge on an ion has the signed infinity
of its Coulomb term, an LJ sphere on an atom the overlap's +Inf, and the other points
of the same wave keep their finite energies.

A tile whose smallest distance has no finite reciprocal is evaluated again, so the
finite energies are compared with those of a grid that has no point on an atom: its
points next to the atoms are the same ones.
"""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu

L = 40.0


def _grid(pm, probe, shift, precision):
    """Energies at 0, 1/16, .., 1 of the first axis; atoms + at 0 and - at 1/2 of it,
    moved off the line by `shift` (a fraction of the third axis)."""
    ff = pm.LJForceField("t", {"A": 3.0, "B": 3.0, "P": 3.4}, {"A": 50.0, "B": 50.0, "P": 120.0}, 12.0)
    box = pm.Box(L, L, L, math.pi / 2, math.pi / 2, math.pi / 2)
    x = pm.Crystal("pair", box, ["A", "B"], np.array([[0.0, 0.5], [0.0, 0.0], [shift, shift]]), atom_q=[1.0, -1.0])
    return pm.energy_grid(x, probe, ff, resolution=(17, 1, 1), units="K", verbose=False, precision=precision,
                          electrostatics=probe.n_charges > 0).data.ravel(order="F")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_points_on_atoms(pm, precision):
    say(f"case: 17 grid points, three of them on atoms ({precision})")
    on = np.zeros(17, dtype=bool)
    on[[0, 8, 16]] = True
    for q in (1.0, -1.0):
        e = _grid(pm, pm.point_charge(q), 0.0, precision)
        np.testing.assert_array_equal(e[on], np.array([q, -q, q]) * math.inf)
        assert np.isfinite(e[~on]).all()
        # 1e-9 of 40 A off the line: energies 2.5 A away change by 1e-16 of themselves
        near = _grid(pm, pm.point_charge(q), 1e-9, precision)
        np.testing.assert_allclose(e[~on], near[~on], rtol=0, atol=(1e-10 if precision == "fp64" else 1e-5) *
                                   np.abs(near[~on]).max())
    e = _grid(pm, pm.lj_sphere("P"), 0.0, precision)
    near = _grid(pm, pm.lj_sphere("P"), 1e-9, precision)
    assert (e[on] == math.inf).all() and (near[on] == math.inf).all()
    np.testing.assert_allclose(e[~on], near[~on], rtol=1e-12 if precision == "fp64" else 2e-6, atol=0)
