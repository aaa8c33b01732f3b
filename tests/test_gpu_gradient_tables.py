"""Gradient runs on the all-atoms path, whose workgroups keep a tile of atoms in
LDS behind the LJ table and the fold constants of every (type, site): tables of
odd and even length in both precisions, against the dual-number oracle with the
bounds of tests/test_gpu_adjoint.py.

A framework keeps image lists of eight radii; a force field of a ninth cutoff
takes the all-atoms path, which evaluates every replicated atom for every site.
"""
import numpy as np
import pytest

from _parity import say
from test_gpu_adjoint import N_BLOCKS, _dual_check, _handles

pytestmark = pytest.mark.gpu

NB = 300


@pytest.mark.parametrize("n_species,probe", [(5, "CO2"), (5, "CH4"), (1, "CH4"), (4, "CO2")])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_all_atoms_gradients_with_tables_of_any_length(pm, orc, precision, n_species, probe):
    case = pm.synthetic.co2_widom_case(seed=60 + n_species, n_species=n_species)
    case.probes["CH4"] = pm.lj_sphere("CH4")
    h = _handles(pm, case, probe)
    _, fw, ew, pr = h
    ff = case.ljff
    for i in range(8):
        short = pm.LJForceField(ff.name, ff.pure_sigma, ff.pure_epsilon, 6.0 + 0.5 * i, ff.mixing_rules)
        pm.device.widom(fw, short, None, pm.device.probe(pm.lj_sphere("CH4"), short), 298.0, 1, 1, 1, precision)
    say(f"case: all-atoms gradients, {n_species} species, {probe} ({precision})")
    _dual_check(pm, orc, h, precision, NB, 61, probe)
    sites = 3 if probe == "CO2" else 1
    n_rep = case.crystal.n_atoms * int(np.prod(pm.replication_factors(case.crystal.box, ff)))
    assert pm.device.last_pair_kernel_stats()[1] == N_BLOCKS * NB * sites * n_rep
