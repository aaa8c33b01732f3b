"""The Fourier part of a point from the folded coefficients, against the plain
sum over the k-vectors, for every range of the third index that has a kernel of
its own (up to 4, 6, 8, 10, 12 and beyond), with empty and one-entry rows.

The k-vectors are drawn at random from the half space (so rows of every length,
gaps and rows with one sign only occur) with random weights of order 10^6 K,
beside which the rounding of the real-space part, which a run with zero weights
takes off, does not count; single ions are compared per insertion.  Tolerance, of
the sum of magnitudes S: phases carry 2 pi m 2^-53 (the three indices together
below 26), on either side, and the recurrences of the cosines 2 m 2^-53; the sum of
some 500 terms sqrt(500) 2^-53: (2 x 164 + 52 + 23) 1.1e-16 = 4.5e-14.
"""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu


def _kvectors(rng, M):
    """Half of the half space's vectors within M, the corner included."""
    m = np.array([(a, b, c) for a in range(M[0] + 1) for b in range(-M[1], M[1] + 1) for c in range(-M[2], M[2] + 1)
                  if a > 0 or b > 0 or (b == 0 and c > 0)])
    keep = rng.random(len(m)) < 0.5
    keep[-1] = True
    return m[keep].astype(np.int32)


@pytest.mark.parametrize("M", [(0, 0, 1), (2, 0, 4), (0, 3, 5), (3, 2, 6), (2, 4, 7), (4, 1, 8), (2, 2, 10), (1, 2, 11),
                               (2, 1, 12), (1, 1, 13), (1, 2, 19)])
def test_fourier_part_of_random_kvector_sets(pm, orc, M):
    say(f"case: k-vectors within {M}")
    rng = np.random.default_rng(sum(M))
    ff = pm.LJForceField("t", {"A": 3.0}, {"A": 50.0}, 6.0)
    box = pm.Box(14.0, 15.0, 16.0, math.pi / 2, 1.4, 1.5)
    x = pm.Crystal("ions", box, ["A"] * 6, rng.random((3, 6)), atom_q=np.array([1.0, -1.0, 0.5, -0.5, 0.25, -0.25]))
    k = _kvectors(rng, M)
    wt = 1e6 * rng.random(len(k))
    fw, pr = pm.device.framework(x, ff), pm.device.probe(pm.point_charge(1.0), ff)

    def energies(wt):
        ep = pm.EwaldParams(tuple(M), 0.3, 6.0, k, wt)
        ew = pm.device.ewald(x, fw, ep)
        return pm.device.widom(fw, ff, ew, pr, 298.0, 9, 1, 200, "fp64", return_energies=True)[1][:, 1]

    got = energies(wt) - energies(np.zeros(len(k)))  # the real-space part drops out
    u = np.array([orc.insertion_uniforms(9, g)[:3] for g in range(200)])
    want = np.zeros(200)
    for xc, q in zip(np.asarray(x.xf).T, x.atom_q):
        want += q * (np.cos(2.0 * np.pi * ((xc - u) @ k.T)) @ wt)
    err = np.abs(got - want).max() / (wt.sum() * np.abs(x.atom_q).sum())
    say(f"   {len(k)} vectors: largest error {err:.2e} of the sum of magnitudes")
    assert err <= 4.5e-14
