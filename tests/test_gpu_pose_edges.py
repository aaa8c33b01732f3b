"""The pose kernels at the edges of their queues and filters: frameworks of 0, 1,
63 to 65 and 255 to 257 atoms (lanes, waves and rounds of a workgroup), every
site count, positions far outside the box, a box narrower than the cutoff sphere
(nearest image only, as the reference), pairs just inside and outside the cutoff,
and k-vector sets whose phases do not fit in LDS, against plain FP64 sums.

Tolerances: FP64 sums of at most 8 x 257 pairs and 2000 k-vectors, each term
good to 1e-13 of itself (a coordinate of a 40 A box carries 1e-14 of itself, the
twelfth power 12 times that): 1e-11 of the sum of the terms' magnitudes.  Mixed:
FP32 terms, 2e-6 of the same sum (1/r^2 to an ulp, six powers, and the erfc fit's
1.2e-7).  Forces are FP64 in both, but a mixed run keeps its LJ constants in
FP32: sigma^2 enters to the sixth power, 4 eps once, 7 x 2^-24 = 4.2e-7 of a
term, and 5e-7 of the sum of the forces' magnitudes.
"""
import math

import numpy as np
import pytest
from scipy.special import erfc

from _parity import say

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-11, "mixed": 2e-6}


def _reference(pm, x, ff, ep, species, q, xf, r_cut):
    """vdw, sr, lr, their magnitudes, dE/dx of poses xf (n, s, 3) and its magnitude."""
    f = x.box.f_to_c
    d = x.xf.T[None, None, :, :] - xf[:, :, None, :]
    d = (d - np.rint(d)) @ f.T
    r2 = (d ** 2).sum(-1)
    kinds = [ff.index(s) for s in x.species]
    lj = np.zeros(r2.shape)
    fl = np.zeros(r2.shape)
    mag = np.zeros(len(xf))
    inside = r2 < r_cut ** 2
    for s, sp in enumerate(species):
        if sp < 0 or not kinds:
            continue
        u = (ff.sigma2_table[kinds, sp][None, :] / r2[:, s]) ** 3
        e = 4.0 * ff.epsilon_table[kinds, sp][None, :]
        lj[:, s] = np.where(inside[:, s], e * u * (u - 1.0), 0.0)
        fl[:, s] = np.where(inside[:, s], 6.0 * e * u * (2.0 * u - 1.0) / r2[:, s], 0.0)
        mag += np.where(inside[:, s], e * u * (u + 1.0), 0.0).sum(-1)
    r = np.sqrt(r2)
    qa = x.atom_q[None, None, :]
    qs = np.asarray(q)[None, :, None]
    t = np.where(inside, qa * erfc(ep.alpha * r) / r, 0.0)
    sr = qs * t / pm.FOUR_PI_EPS0
    fc = np.where(inside, qs * (t + qa * 2.0 * ep.alpha / math.sqrt(math.pi) * np.exp(-(ep.alpha * r) ** 2)) / r2, 0.0)
    g = ((fl + fc / pm.FOUR_PI_EPS0)[..., None] * d).sum(2)
    gm = ((np.abs(fl) + np.abs(fc) / pm.FOUR_PI_EPS0) * r).sum((1, 2))
    ph = 2.0 * math.pi * ep.kidx @ x.xf
    A = ep.wt * ((x.atom_q * np.exp(1j * ph)).sum(1) if x.n_atoms else 0.0)
    th = 2.0 * math.pi * xf @ ep.kidx.T
    lr = np.asarray(q)[None, :] * (A.real * np.cos(th) + A.imag * np.sin(th)).sum(-1)
    dk = 2.0 * math.pi * np.asarray(q)[None, :, None] * ((A.imag * np.cos(th) - A.real * np.sin(th)) @ ep.kidx)
    g = g + dk @ x.box.c_to_f
    gm = gm + np.abs(dk).sum((1, 2)) * np.abs(x.box.c_to_f).max() + np.abs(A).sum()
    over = (r2 < 0.1) & inside
    over[:, [s for s, sp in enumerate(species) if sp < 0], :] = False
    vdw = np.where(over.any((1, 2)), np.inf, lj.sum((1, 2)))
    return vdw, sr.sum((1, 2)), lr.sum(1), mag, np.abs(sr).sum((1, 2)), np.abs(lr).sum(1) + np.abs(A).sum(), g, gm


def _system(pm, n, edge, r_cut, seed):
    rng = np.random.default_rng(seed)
    ff = pm.LJForceField("t", {"A": 3.0, "B": 3.4, "P": 3.2}, {"A": 50.0, "B": 70.0, "P": 90.0}, r_cut)
    box = pm.Box(edge, 1.1 * edge, 0.95 * edge, math.radians(85.0), math.radians(97.0), math.radians(101.0))
    x = pm.Crystal("pose_edges", box, ["AB"[k] for k in rng.integers(0, 2, n)], rng.random((3, n)) - 0.3,
                   rng.uniform(-0.7, 0.7, n))
    return rng, ff, x


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,edge,r_cut,ns,reach,kmax", [
    (0, 30.0, 12.8, 1, 1.0, None), (1, 30.0, 12.8, 2, 1.0, None), (63, 30.0, 12.8, 3, 3.0, None),
    (64, 30.0, 12.8, 4, 1.0, None), (65, 30.0, 12.8, 5, 200.0, None), (255, 31.0, 12.8, 6, 1.0, None),
    (256, 31.0, 12.0, 8, 1.0, None), (257, 31.0, 12.8, 3, 1.0, None), (257, 14.0, 12.8, 3, 1.0, None),
    (80, 27.0, 9.0, 3, 1.0, 800)])
def test_pose_energies_and_forces(pm, precision, n, edge, r_cut, ns, reach, kmax):
    say(f"case: {n} atoms, {ns} sites, edge {edge} A, r_c {r_cut} A, k-vectors {kmax} ({precision})")
    rng, ff, x = _system(pm, n, edge, r_cut, 7 * n + ns)
    ep = pm.setup_Ewald_sum(x.box, r_cut)
    if kmax is not None:  # phases of 800 + 3 powers per site: more than the kernel keeps
        k = np.stack([np.array([1, 3, 790]), np.array([0, -2, 5]), np.array([kmax, -7, 2])], axis=1).astype(np.int32)
        ep = pm.EwaldParams((1, 1, 1), ep.alpha, ep.sr_cutoff_r, k, np.array([1.0, 2.0, 0.5]))
    poses = (rng.random((37, 1, 3)) - 0.5) * 2.0 * reach + 0.05 * rng.normal(size=(37, ns, 3))
    species = [ff.index("P") if s % 3 != 2 else -1 for s in range(ns)]
    q = [0.4 * (-1) ** s if s % 4 != 1 else 0.0 for s in range(ns)]
    fw, ew = pm.device.framework(x, ff), None
    ew = pm.device.ewald(x, fw, ep)
    e, g = pm.device.pose_gradients(fw, ff, ew, species, q, poses, precision)
    vdw, sr, lr, m_lj, m_sr, m_lr, gw, gm = _reference(pm, x, ff, ep, species, q, poses, r_cut)
    np.testing.assert_array_equal(np.isinf(e[:, 0]), np.isinf(vdw))
    ok = np.isfinite(vdw)
    tol = TOL[precision]
    far = max(1.0, reach)  # a position of `far` boxes is off by that many ulp
    assert np.all(np.abs(e[ok, 0] - vdw[ok]) <= tol * far * (m_lj[ok] + 1e-6))
    assert np.all(np.abs(e[:, 1] - sr) <= tol * far * (m_sr + 1e-6))
    assert np.all(np.abs(e[:, 2] - lr) <= 1e-11 * far * (m_lr + 1e-6) * (1.0 if kmax is None else 100.0))
    if n == 0 or kmax is not None:
        return
    tol_g = 1e-11 if precision == "fp64" else 5e-7
    assert np.all(np.abs(g - gw).max(axis=(1, 2))[ok] <= tol_g * far * (gm[ok] + 1e-6))
    # the energy-only kernels agree with the forces' kernel
    lj_sites = [s for s in range(ns) if species[s] >= 0]
    v = pm.vdw_energies(x, ["P"] * len(lj_sites), poses[:, lj_sites], ff, precision=precision)
    np.testing.assert_allclose(v[ok], e[ok, 0], rtol=0, atol=float(tol * far * (m_lj[ok].max() + 1e-6)))
    s2, l2 = pm.electrostatic_energies(x, q, poses, ep, precision=precision)
    np.testing.assert_allclose(s2, e[:, 1], rtol=0, atol=float(tol * far * (m_sr.max() + 1e-6)))
    np.testing.assert_allclose(l2, e[:, 2], rtol=0, atol=float(1e-11 * far * (m_lr.max() + 1e-6)))
