"""Small launches share the image list of 64 points out over 2, 8 or 16 waves; a
point's energies are the same bit for bit whichever kernel takes them, because
the FP64 sums run over fixed parts of the list in fixed order.

The first insertions of a run of one block do not depend on its length, so runs
of growing length, each on another side of the rule (192 and 1024 waves of 64
points), must agree on them exactly.  The two-atom framework has fewer tiles
than parts; lengths of 1, 64 and 65 leave most of the waves without points.
"""
import math

import numpy as np
import pytest

from _parity import say
from test_gpu_batch import _handles

pytestmark = pytest.mark.gpu

SIZES = {"CH4": (1, 64, 65, 10_000, 10_500, 40_700, 41_200, 65_200, 65_800, 114_400, 115_000),
         "CO2": (1, 65, 3_300, 3_500, 13_500, 13_800, 21_700, 22_000, 38_100, 38_400)}


@pytest.mark.parametrize("name", ["CH4", "CO2"])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_insertion_energies_do_not_depend_on_the_split(pm, precision, name):
    say(f"case: {name} insertions, runs of {SIZES[name]} ({precision})")
    case = pm.synthetic.lj_grid_case() if name == "CH4" else pm.synthetic.co2_widom_case()
    fw, ff, ew, pr, _ = _handles(pm, case, name)
    en = {n: pm.device.widom(fw, ff, ew, pr, 298.0, 5, 1, n, precision, return_energies=True)[1] for n in SIZES[name]}
    full = en[SIZES[name][-1]]
    assert np.isfinite(full).any() and np.isinf(full[:, 0]).any()
    for n, e in en.items():
        np.testing.assert_array_equal(e, full[:n], err_msg=str(n))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_list_of_fewer_tiles_than_parts(pm, precision):
    say(f"case: CH4 in two atoms of a 40 A box ({precision})")
    ff = pm.LJForceField("t", {"A": 3.0, "CH4": 3.4}, {"A": 50.0, "CH4": 120.0}, 6.0)
    x = pm.Crystal("pair", pm.Box(40.0, 40.0, 40.0, math.pi / 2, math.pi / 2, math.pi / 2), ["A", "A"],
                   np.array([[0.1, 0.6], [0.2, 0.5], [0.3, 0.5]]))
    fw, pr = pm.device.framework(x, ff), pm.device.probe(pm.lj_sphere("CH4"), ff)
    en = [pm.device.widom(fw, ff, None, pr, 298.0, 5, 1, n, precision, return_energies=True)[1]
          for n in (1000, 20_000, 50_000, 120_000)]
    assert (en[0] != 0.0).any()
    for e in en[:-1]:
        np.testing.assert_array_equal(e, en[-1][:len(e)])
