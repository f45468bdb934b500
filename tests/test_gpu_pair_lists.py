"""The tiles' pair lists and their three classes of pairs (two bare charges, one,
none), at compositions and sizes that the water boxes do not reach.

Boxes of 200 sites (four blocks, the last of eight) on a lattice, half of them
unjittered so that separations lie exactly along x, in which all, none or a
random half of the sites are bare charges, against the FP64 oracle converged to
1e-10 Debye.  The FP64 path at 1e-9 Debye: forces within 1e-7 relative RMS (first
order in the residual, 1e-8 of the dipoles).  The mixed path: 2e-5, that is
thirty roundings of 2^-24 in a pair and a factor ten for the cancellation
among a lattice site's neighbours.

A box of 20,000 general sites (313 blocks of about 6,000 general pairs each, more
than one queue of the FP64 kernel holds; groups of two tiles in the mixed path):
the forces of the two paths, whose kernels differ, agree to the same 2e-5.

The energy gradients of covalent partners that lie exactly along x, beside others
that do not: displaced by 1e-7 nm across x, every gradient must stay within
1e-5 of the largest of its class (they vary over the bond length, 0.1 nm, so the
displacement moves them by about 1e-6).
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import ewald_alpha, random_traceless_octopole, random_traceless_quadrupole
from oracle import oracle

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum())


def lattice_box(n, bare_fraction, spacing, seed, cutoff, grid):
    """n sites of alternating charge on a cubic lattice; every second one is
    jittered, and a random bare_fraction are charges only."""
    rng = np.random.default_rng(seed)
    k = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    cells = np.array([(x, y, z) for x in range(k) for y in range(k) for z in range(k)])[:n]
    pos = (cells + 0.5) * spacing
    pos[1::2] += rng.uniform(-0.03, 0.03, size=pos[1::2].shape)
    order = rng.permutation(n)
    bare = np.zeros(n, dtype=bool)
    bare[order[:int(round(bare_fraction * n))]] = True
    force = MPIDForce()
    charge = 0.4 * (-1.0) ** cells.sum(1)
    charge -= charge.mean()
    for a in range(n):
        dip = [0.0] * 3 if bare[a] else list(rng.normal(0.0, 0.005, 3))
        quad = [0.0] * 6 if bare[a] else random_traceless_quadrupole(rng, 1e-4)
        octo = [0.0] * 10 if bare[a] else random_traceless_octopole(rng, 1e-5)
        alpha = [0.0] * 3 if bare[a] else [0.0005] * 3
        force.addMultipole(float(charge[a]), dip, quad, octo, MPIDForce.NoAxisType, -1, -1, -1, 1.3, alpha)
    force.setDefaultTholeWidth(5.0)
    force.setPolarizationType(MPIDForce.Mutual)
    force.setMutualInducedMaxIterations(60)
    force.setNonbondedMethod(MPIDForce.PME)
    force.setCutoffDistance(cutoff)
    force.setPMEParameters(ewald_alpha(cutoff), grid, grid, grid)
    return force, pos, np.full(3, k * spacing)


def forces(force, pos, box, precision, eps):
    force.setMutualInducedTargetEpsilon(eps)
    k = HipCalcMPIDForceKernel(precision)
    k.initialize(len(pos), force, default_box=box)
    return k.execute(pos, box)[1]


@pytest.mark.parametrize("bare_fraction", [0.0, 0.5, 1.0])
def test_classes_of_pairs(bare_fraction):
    force, pos, box = lattice_box(200, bare_fraction, 0.32, 11, 0.9, 24)
    force.setMutualInducedTargetEpsilon(1e-10)
    ref = oracle.evaluate(force.flatten(), pos, box)["forces"]
    for precision, eps, tol in (("double", 1e-9, 1e-7), ("mixed", 1e-6, 2e-5)):
        print(f"[gpu] 200 sites, {bare_fraction} bare, {precision}", flush=True)
        assert rel_rms(forces(force, pos, box, precision, eps), ref) <= tol


def test_many_general_pairs():
    force, pos, box = lattice_box(20000, 0.0, 0.25, 12, 0.9, 90)
    print("[gpu] 20000 general sites", flush=True)
    double = forces(force, pos, box, "double", 1e-6)
    assert rel_rms(forces(force, pos, box, "mixed", 1e-6), double) <= 2e-5


def test_gradients_of_partners_along_x():
    rng = np.random.default_rng(13)
    pos = np.array([[0.0, 0.0, 0.0], [0.1, 0.0, 0.0], [0.02, 0.4, 0.03], [0.07, 0.47, 0.06]])
    force = MPIDForce()
    for a in range(4):
        force.addMultipole(0.3 * (-1.0) ** a, list(rng.normal(0.0, 0.005, 3)), random_traceless_quadrupole(rng, 1e-4),
                           random_traceless_octopole(rng, 1e-5), MPIDForce.NoAxisType, -1, -1, -1, 1.3, [0.0005] * 3)
    for a, b in ((0, 1), (2, 3)):
        force.setCovalentMap(a, MPIDForce.Covalent14, [b])
        force.setCovalentMap(b, MPIDForce.Covalent14, [a])
    force.set14ScaleFactor(0.5)
    force.setDefaultTholeWidth(5.0)
    force.setPolarizationType(MPIDForce.Mutual)
    force.setMutualInducedTargetEpsilon(1e-9)
    k = HipCalcMPIDForceKernel("double")
    k.initialize(4, force)
    print("[gpu] gradients of partners along x", flush=True)
    on = k.energyGradients(pos, None, all_sites=True)
    off = pos.copy()
    off[1, 1] += 1e-7
    near = k.energyGradients(off, None, all_sites=True)
    for name in ("positions", "charges", "dipoles", "quadrupoles", "octopoles", "polarity"):
        a, b = np.asarray(on[name]), np.asarray(near[name])
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max(), name
