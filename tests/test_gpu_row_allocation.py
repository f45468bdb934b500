"""A context whose list buffers could not be allocated can be used again.

720,000 charges squeezed into 1.9 nm: most of the 11,250 blocks are within the
0.9 nm cutoff of each other, and the pair lists of their tiles would take 470 GB
(8 KB each), more than the 288 of the card.  300,000 in 1.84 nm: the pair lists fit
(80 GB), the neighbour lists of 190,000 entries an atom (230 GB) do not.  Both
evaluations end in an error before a list is built.  The same context at an
ordinary density then gives what a fresh one gives: the same kernels on the same
inputs, 1e-9 relative in the energy and 1e-6 in the forces for the order of the
sums on the grid.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import ewald_alpha

pytestmark = pytest.mark.gpu


class ManyCharges(MPIDForce):
    """n charges of alternating sign, from one pair's flat arrays."""

    def __init__(self, n):
        super().__init__()
        for charge in (0.2, -0.2):
            self.addMultipole(charge, [0.0] * 3, [0.0] * 6, [0.0] * 10, MPIDForce.NoAxisType, -1, -1, -1, 1.3, [0.0] * 3)
        self.n = n

    def getNumMultipoles(self):
        return self.n

    def flatten(self):
        flat = super().flatten()
        for name in ("charges", "dipoles", "quadrupoles", "octopoles", "axis_types", "atom_z", "atom_x", "atom_y",
                     "tholes", "polarity"):
            flat[name] = np.tile(flat[name], self.n // 2)
        flat["cov_offsets"] = np.zeros(4 * self.n + 1, dtype=np.int32)
        flat["n"] = self.n
        return flat


@pytest.mark.parametrize("n,cells,squeeze", [(720000, 90, 0.1), (300000, 67, 0.13)], ids=["rows", "lists"])
def test_context_after_a_failed_allocation(n, cells, squeeze):
    edge = cells * (19.0 / 90)
    sites = np.indices((cells,) * 3).reshape(3, -1).T[:n]
    pos = (sites + 0.5) * (19.0 / 90) + np.random.default_rng(7).uniform(-0.05, 0.05, size=(n, 3))
    box = np.full(3, edge)
    force = ManyCharges(n)
    force.setNonbondedMethod(MPIDForce.PME)
    force.setPolarizationType(MPIDForce.Direct)
    force.setCutoffDistance(0.9)
    force.setPMEParameters(ewald_alpha(0.9), 96, 96, 96)
    k = HipCalcMPIDForceKernel("mixed")
    k.initialize(n, force)
    print("[gpu] an allocation beyond the card's memory", flush=True)
    with pytest.raises(RuntimeError, match="memory"):
        k.execute(squeeze * pos, squeeze * box)
    print("[gpu] the same context at an ordinary density", flush=True)
    e1, f1 = k.execute(pos, box)
    fresh = HipCalcMPIDForceKernel("mixed")
    fresh.initialize(n, force)
    e2, f2 = fresh.execute(pos, box)
    assert abs(e1 - e2) <= 1e-9 * abs(e2)
    assert np.sqrt(((f1 - f2) ** 2).sum() / (f2 ** 2).sum()) <= 1e-6
