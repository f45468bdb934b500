"""Rounding of the real-space force sums in FP64.

A cluster of 2,000 sites with moments, no polarisability and no cutoff: every
pair is a general one, and the force on a site is a sum over its block's tiles.
The fixed-point accumulators take a value truncated to 2^-32.  Kept in FP64 until
a tile is done, a component takes at most 2 (blocks + 1) such values from the
tiles (the charge-charge channel and the rest) and one per split of its block
row: 2 x 33 + 16, each off by a fraction of a unit that is uniform in [0, 1), so
that the RMS error is at most sqrt(82 / 3) = 5.2 units; FP64 rounding of forces of
1e3 adds 0.02.  Within 8 units of the FP64 oracle, where a truncation per pair
gives sqrt(1000 / 3) = 18.  (RMS over 6,000 components: its own spread is 1%.)
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import random_traceless_octopole, random_traceless_quadrupole
from oracle import oracle

pytestmark = pytest.mark.gpu


def test_general_pairs_are_summed_in_fp64():
    rng = np.random.default_rng(31)
    cells = np.array([(x, y, z) for x in range(13) for y in range(13) for z in range(13)])[:2000]
    pos = 0.3 * cells + rng.uniform(-0.03, 0.03, size=(2000, 3))
    force = MPIDForce()
    for a in range(2000):
        force.addMultipole(0.4 * (-1.0) ** cells[a].sum(), list(rng.normal(0.0, 0.005, 3)),
                           random_traceless_quadrupole(rng, 1e-4), random_traceless_octopole(rng, 1e-5),
                           MPIDForce.NoAxisType, -1, -1, -1, 1.3, [0.0] * 3)
    force.setNonbondedMethod(MPIDForce.NoCutoff)
    force.setPolarizationType(MPIDForce.Direct)
    ref = oracle.evaluate(force.flatten(), pos, None)["forces"]
    k = HipCalcMPIDForceKernel("double")
    k.initialize(2000, force)
    print("[gpu] force sums of 2000 general sites", flush=True)
    error = k.execute(pos, None)[1] - ref
    print(f"[gpu] RMS error {np.sqrt((error ** 2).mean()) * 2.0 ** 32:.2f} units", flush=True)
    assert np.sqrt((error ** 2).mean()) <= 8.0 * 2.0 ** -32
