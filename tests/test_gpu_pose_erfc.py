"""The real-space Ewald term of explicit poses over the splitting parameters that
an Ewald handle accepts: alpha r_c on both sides of 3.68, where the kernels change
from their table of erfc to the function, and far beyond it (a table's error at
alpha r_c = 20 is larger than the term).

One atom of charge 1 in a 40 A box, poses of one charge at distances up to the
cutoff, energies and forces against math.erfc.

Tolerances.  Positions of a 40 A box carry 9e-15 A, so r >= 0.5 A is good to 2e-14
of itself and erfc(x), whose logarithm changes by at most 2 x^2 + 2 per relative
change of x, to (2 x^2 + 2) 2e-14 of itself; 1/r and the products add less: (2 x^2
+ 4) 2e-14 of the term.  The table may add its truncation, half an ulp of 1, and as
much again for the rounding of its coefficients and its Horner steps: 4e-16 / r.
"""
import math

import numpy as np
import pytest

from _parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha_rc", [1.0, 3.0, 3.67, 3.70, 5.0, 8.0, 20.0])
def test_real_space_term_for_any_splitting_parameter(pm, alpha_rc):
    say(f"case: one charge, 400 distances, alpha r_c = {alpha_rc}")
    r_c, edge = 12.0, 40.0
    ff = pm.LJForceField("t", {"A": 3.0}, {"A": 50.0}, r_c)
    box = pm.Box(edge, edge, edge, math.pi / 2, math.pi / 2, math.pi / 2)
    x = pm.Crystal("one", box, ["A"], np.array([[0.25], [0.5], [0.75]]), atom_q=[1.0])
    alpha = alpha_rc / r_c
    ep = pm.EwaldParams((1, 1, 1), alpha, r_c, np.array([[1, 0, 0]], dtype=np.int32), np.array([0.0]))
    fw = pm.device.framework(x, ff)
    ew = pm.device.ewald(x, fw, ep)
    r = np.linspace(0.5, r_c - 1e-3, 400)
    rng = np.random.default_rng(3)
    u = rng.normal(size=(400, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    xf = x.xf[:, 0] + u * r[:, None] / edge
    d = (x.xf[:, 0] - xf) * edge
    r = np.linalg.norm(d, axis=1)
    q = 0.7
    ec = np.array([math.erfc(alpha * v) for v in r])
    want = q * ec / r / pm.FOUR_PI_EPS0
    f = q * (ec / r + 2.0 * alpha / math.sqrt(math.pi) * np.exp(-(alpha * r) ** 2)) / r ** 2 / pm.FOUR_PI_EPS0
    rel = (2.0 * (alpha * r) ** 2 + 4.0) * 2e-14
    table = 4e-16 / r * q / pm.FOUR_PI_EPS0 if alpha_rc < 3.68 else 0.0
    e, g = pm.device.pose_gradients(fw, None, ew, [-1], [q], xf[:, None, :], "fp64")
    sr, _ = pm.electrostatic_energies(x, [q], xf[:, None, :], ep, precision="fp64")
    for name, got in (("energies", sr), ("energies with forces", e[:, 1])):
        over = np.abs(got - want) / (rel * want + table)
        say(f"   {name}: largest error {over.max():.2f} of the bound, at alpha r = {(alpha * r)[over.argmax()]:.2f}")
        assert over.max() <= 1.0
    err = np.abs(g[:, 0, :] - f[:, None] * d).max(axis=1)
    over = err / (2.0 * rel * f * r + table / r + 1e-300)
    say(f"   forces: largest error {over.max():.2f} of the bound")
    assert over.max() <= 1.0
    # mixed energies are FP32 terms, their forces FP64
    gm = pm.device.pose_gradients(fw, None, ew, [-1], [q], xf[:, None, :], "mixed")[1]
    np.testing.assert_array_equal(gm, g)
