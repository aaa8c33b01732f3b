"""Widom runs in unit cells so large that a cell of a run holds a few points or
none.  The number of waves that share the image list follows the workgroups with
points, not the points alone.

The first insertions of a run of one block do not depend on its length, so their
energies must be the same bit for bit in runs of growing length: 16 waves (27
cells of a 21 A box), 8 (216 cells of 40 A), 4 (1000 cells of 60 A) and one, and
the candidate pairs counted must not depend on the waves that found them: a run
with every insertion in one wave of a workgroup of four, or of sixteen, counts
each once.  A batch of 17 runs of 64,000 cells each, with one insertion per
block, takes a launch's work-items to their limit if every cell gets a workgroup
of 1024 for each quarter of a slice.
"""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu


def _large(pm, edge, n, seed=5):
    rng = np.random.default_rng(seed)
    ff = pm.LJForceField("t", {"A": 3.0, "B": 3.4, "CH4": 3.7}, {"A": 50.0, "B": 70.0, "CH4": 148.0}, 9.0)
    box = pm.Box(edge, edge, edge, math.pi / 2, math.pi / 2, math.pi / 2)
    x = pm.Crystal("large", box, ["AB"[k] for k in rng.integers(0, 2, n)], rng.random((3, n)))
    xr = pm.replicate(x, pm.replication_factors(box, ff))
    return pm.device.framework(xr, ff), ff, pm.device.probe(pm.lj_sphere("CH4"), ff)


@pytest.mark.parametrize("edge,n", [(21.0, 200), (40.0, 1500), (60.0, 4000)])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_sparse_insertion_energies_do_not_depend_on_the_waves(pm, precision, edge, n):
    say(f"case: CH4 in {n} atoms of a {edge} A cell, runs of growing length ({precision})")
    fw, ff, pr = _large(pm, edge, n)
    lengths = (1, 40, 1000, 5000, 20_000, 90_000, 400_000)
    en = {k: pm.device.widom(fw, ff, None, pr, 298.0, 9, 1, k, precision, return_energies=True)[1] for k in lengths}
    full = en[lengths[-1]]
    assert np.isfinite(full[:, 0]).any() and np.isinf(full[:, 0]).any()
    for k, e in en.items():
        np.testing.assert_array_equal(e, full[:k], err_msg=str(k))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_candidates_are_counted_once(pm, precision):
    say(f"case: one insertion's candidate pairs, alone and among others ({precision})")
    fw, ff, pr = _large(pm, 60.0, 4000)
    # one wave holds the one point: its sphere is the point, its candidates the images within the cutoff of it
    pm.device.widom(fw, ff, None, pr, 298.0, 9, 1, 1, precision)
    alone = pm.device.last_pair_kernel_stats()[1]
    fw2, ff2, pr2 = _large(pm, 21.0, 171)  # the same density
    pm.device.widom(fw2, ff2, None, pr2, 298.0, 9, 1, 1, precision)
    small = pm.device.last_pair_kernel_stats()[1]
    expect = 4000 / 60.0 ** 3 * 4.0 / 3.0 * math.pi * 9.0 ** 3  # 57 in a sphere of the cutoff
    assert 0.4 * expect < alone < 2.0 * expect and 0.4 * expect < small < 2.0 * expect


def test_batch_of_runs_with_more_cells_than_a_launch_has_groups(pm):
    say("case: 17 runs of 5 x 1 insertions in a 275 A cell, mixed")
    fw, ff, pr = _large(pm, 275.0, 40)
    ffh = pm.device.forcefield(ff)
    runs = [(fw, ffh, None, pr, 298.0, 100 + k, 5, 1) for k in range(17)]
    got = pm.device.widom_batch(runs, "mixed")
    for run, g in zip(runs, got):
        assert np.array_equal(g, pm.device.widom(*run, "mixed"))
