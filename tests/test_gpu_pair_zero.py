"""Points with no charge inside the real-space cutoff: their real-space energy is
zero, in both precisions, on the image-list and the all-atoms path, and so is the
charge derivative of a run of such points.

The framework's two ions and its handle (one k-vector of weight zero) leave nothing
but the real-space part; most of a 40 A cell is beyond the 6 A cutoff of either.
"""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("all_atoms", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_no_charge_in_reach_is_zero_energy(pm, precision, all_atoms):
    say(f"case: ion in two ions of a 40 A cell ({precision}, {'all atoms' if all_atoms else 'image list'})")
    r_c = 6.0
    ff = pm.LJForceField("t", {"A": 3.0, "B": 3.0}, {"A": 50.0, "B": 50.0}, r_c)
    box = pm.Box(40.0, 40.0, 40.0, math.pi / 2, math.pi / 2, math.pi / 2)
    x = pm.Crystal("pair", box, ["A", "B"], np.array([[0.2, 0.3], [0.2, 0.2], [0.2, 0.2]]), atom_q=[1.0, -1.0])
    fw = pm.device.framework(x, ff)
    ew = pm.device.ewald(x, fw, pm.EwaldParams((1, 1, 1), 0.5, r_c, np.array([[1, 0, 0]], dtype=np.int32),
                                               np.array([0.0])))
    probe = pm.device.probe(pm.point_charge(1.0), ff)
    if all_atoms:  # a framework keeps image lists of eight radii
        for i in range(8):
            short = pm.LJForceField("s", {"A": 3.0, "B": 3.0}, {"A": 50.0, "B": 50.0}, 3.0 + 0.25 * i)
            pm.device.widom(fw, short, None, pm.device.probe(pm.lj_sphere("A"), short), 298.0, 1, 1, 1, precision)
    n = 4000
    sums, en = pm.device.widom(fw, ff, ew, probe, 298.0, 11, 1, n, precision, return_energies=True)
    e = en[:, 1]
    zero = e == 0.0
    # two spheres of 6 A, 4 A apart, in the cell: 2.5% of it
    assert 0.95 < zero.mean() < 0.995
    assert np.abs(e[~zero]).min() > 1e-12
    g = pm.device.widom_gradient(fw, ff, ew, probe, 298.0, 11, 1, n, precision, ff)
    np.testing.assert_array_equal(g[0], sums)
