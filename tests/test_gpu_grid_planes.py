"""Sites on the planes of the PME grid and within a few roundings of them.

There an atom's grid coordinate is an integer up to rounding, so its spline
offset is almost 0 at one stencil start or almost 1 at the one before; the spread
charges are the same either way (the splines are continuous), as long as start
and offset belong together.  Grids with owned cores against the untiled spreading
of the FP64 path, which evaluates both once per atom.

FP64: a crystal of sites with moments exactly on planes, boxes whose edges do not
divide exactly, forces with direct polarization within 1e-10 relative RMS (the
order of the sums).  Mixed: the field of random dipoles at sites moved off their
planes by up to 4 units of 2^-24 of the coordinate, within 1e-4 (positions of up to
5 nm in FP32 are off by 3e-7 nm, over the nearest distance of 0.2 nm three times
that relatively, with a factor twenty in hand).  A site at the wrong start moves
its charges by a whole grid spacing.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import ewald_alpha, random_traceless_octopole, random_traceless_quadrupole

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum())


def crystal(edge, n, every, rng):
    """Sites on every `every`-th plane of an n^3 grid, alternating charges and random moments."""
    m = np.indices((n // every,) * 3).reshape(3, -1).T * every
    force = MPIDForce()
    for a in range(len(m)):
        force.addMultipole(0.3 * (-1.0) ** (m[a].sum() // every), list(rng.normal(0.0, 0.005, 3)),
                           random_traceless_quadrupole(rng, 1e-4), random_traceless_octopole(rng, 1e-5),
                           MPIDForce.NoAxisType, -1, -1, -1, 1.3, [0.0005] * 3)
    force.setDefaultTholeWidth(5.0)
    force.setNonbondedMethod(MPIDForce.PME)
    force.setPolarizationType(MPIDForce.Direct)
    force.setCutoffDistance(0.8)
    force.setPMEParameters(ewald_alpha(0.8), n, n, n)
    return force, edge * m / n, np.full(3, edge)


def kernel(precision, tiling, force, pos, box):
    k = HipCalcMPIDForceKernel(precision, spread_tiling=tiling)
    k.initialize(len(pos), force, default_box=box)
    return k


@pytest.mark.parametrize("edge,n,every,level", [(2.97, 40, 4, 2), (2.7, 48, 4, 2), (3.1, 64, 5, 3), (4.966, 64, 4, 3)])
def test_crystal_on_grid_planes(edge, n, every, level):
    force, pos, box = crystal(edge, n, every, np.random.default_rng(n))
    print(f"[gpu] {len(pos)} sites on planes of {n}^3, FP64", flush=True)
    owned = kernel("double", (level, 1), force, pos, box).execute(pos, box)[1]
    untiled = kernel("double", (-1, 0), force, pos, box).execute(pos, box)[1]
    print(f"[gpu] difference {rel_rms(owned, untiled):.1e}", flush=True)
    assert rel_rms(owned, untiled) <= 1e-10


@pytest.mark.parametrize("edge,n,every,level", [(2.97, 40, 4, 2), (4.966, 64, 4, 3)])
def test_sites_next_to_grid_planes(edge, n, every, level):
    rng = np.random.default_rng(n + 1)
    force, pos, box = crystal(edge, n, every, rng)
    pos = pos * (1.0 + rng.integers(-4, 5, size=pos.shape) * 2.0 ** -24)
    mu = rng.normal(0.0, 0.005, size=pos.shape)
    print(f"[gpu] {len(pos)} sites next to planes of {n}^3, mixed", flush=True)
    owned = kernel("mixed", (level, 1), force, pos, box).computeInducedField(pos, box, mu)
    untiled = kernel("double", (-1, 0), force, pos, box).computeInducedField(pos, box, mu)
    print(f"[gpu] difference {rel_rms(owned, untiled):.1e}", flush=True)
    assert rel_rms(owned, untiled) <= 1e-4
