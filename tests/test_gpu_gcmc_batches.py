"""The pair batches of a chain's energies at their edges, against the oracle's chain:
framework sizes around one, two and four atoms per work-item (256 of them), with
and without cell lists (the 46 A box), and more guest sites than work-items.

Tolerances are those of the comparisons with the oracle's chain elsewhere: counts
and decisions equal, energies to 1e-9.
"""
import math

import numpy as np
import pytest

from test_gpu_gcmc import _compare, _oracle_chains, say

pytestmark = pytest.mark.gpu


def _system(pm, n_atoms, length):
    rng = np.random.default_rng(n_atoms)
    ff = pm.LJForceField("t", {"A": 1.2, "B": 1.4, "G": 1.0}, {"A": 30.0, "B": 20.0, "G": 40.0}, 12.8)
    box = pm.Box(length, length, length, math.pi / 2, math.pi / 2, math.pi / 2)
    return ff, pm.Crystal("random", box, ["AB"[i % 2] for i in range(n_atoms)], rng.random((3, n_atoms)))


@pytest.mark.parametrize("n_atoms,length", [(1, 26.0), (255, 26.0), (256, 26.0), (257, 26.0), (511, 26.0), (513, 26.0),
                                            (768, 26.0), (1024, 26.0), (1025, 26.0), (1537, 26.0), (700, 46.0),
                                            (2100, 46.0), (5200, 46.0)])
def test_framework_sizes_match_oracle(pm, orc, n_atoms, length):
    from oracle import gcmc as ogc
    say(f"case: GCMC of one LJ site among {n_atoms} atoms of a {length} A box, 40 cycles")
    ff, x = _system(pm, n_atoms, length)
    g = pm.lj_sphere("G")
    fw = pm.device.framework(x, ff)
    dev = pm.device.GcmcChains(fw, ff, [g], [300.0], [[2e6]], 20, 20, capacity=256, seed=4)
    dev.run(40)
    och = _oracle_chains(ogc, pm, x, ff, [g], [300.0], [[2e6]], 20, 20, 4, 256)
    och[0].run(40)
    _compare(dev, och, 1, n_atoms)


@pytest.mark.parametrize("n_start", [255, 256, 257, 513])
def test_more_guests_than_work_items_match_oracle(pm, orc, n_start):
    from oracle import gcmc as ogc
    say(f"case: GCMC started from {n_start} guests, 2 cycles")
    ff, x = _system(pm, 3, 26.0)
    g = pm.lj_sphere("G")
    fw = pm.device.framework(x, ff)
    i = np.arange(n_start)
    com = (np.stack([i % 9, i // 9 % 9, i // 81], axis=1) + 0.3) / 9.0
    args = ([300.0], [[2e7]], 1, 5)
    dev = pm.device.GcmcChains(fw, ff, [g], *args, capacity=600, seed=4)
    dev.set_molecules(0, 0, com[:, None, :], com)
    dev.run(2)
    och = _oracle_chains(ogc, pm, x, ff, [g], *args, 4, 600)
    och[0].set_molecules(0, com[:, None, :], com)
    och[0].run(2)
    _compare(dev, och, 1, n_start)
