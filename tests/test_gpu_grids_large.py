"""PME grids with the largest splits of the transforms' register steps: 160 =
10 x 16, 192 = 12 x 16 and 256 = 16 x 16 along each axis, in planes that fit a
workgroup's LDS and in ones that do not (256 x 256 and 160 x 192), and in the mixed
path also 72 to 144.

A box of 32 waters against the FP64 oracle on the same grid, converged to 1e-10
Debye.  The FP64 path at 1e-9 Debye: forces within 1e-7 relative RMS (first order
in the residual, 1e-8 of the dipoles; transforms and fixed-point sums are at
1e-13).  The mixed path within 1e-3: its derivatives of the FP32 potential on a
spacing h carry 6e-8 / h^3 times the quadrupoles of 1e-4, about 1e-4 of the forces at
h = 0.004 nm (there are no octopoles, whose noise goes with h^-4), with a
factor ten in hand; an element misplaced or wrongly weighted by a transform
moves the forces by their own size.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.waterbox import _o_parameters, make_small_waterbox
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(160, 18, 24), (20, 160, 27), (24, 25, 160), (192, 16, 20), (15, 192, 24),
                                  (16, 27, 192), (256, 12, 20), (18, 256, 15), (20, 24, 256), (256, 256, 10),
                                  (160, 192, 12), (72, 80, 81), (90, 96, 100), (108, 40, 120), (144, 128, 20)])
def test_large_grid(grid):
    force, pos, box = make_small_waterbox(32, 23, _o_parameters(np.random.default_rng(23), False, True))
    force.setPMEParameters(force.getPMEParameters()[0], *grid)
    force.setMutualInducedTargetEpsilon(1e-10)
    ref = oracle.evaluate(force.flatten(), pos, box)["forces"]
    for precision, eps, tol in (("double", 1e-9, 1e-7), ("mixed", 1e-6, 1e-3)):
        force.setMutualInducedTargetEpsilon(eps)
        k = HipCalcMPIDForceKernel(precision)
        k.initialize(len(pos), force, default_box=box)
        print(f"[gpu] grid {grid} {precision}", flush=True)
        F = k.execute(pos, box)[1]
        error = np.sqrt(((F - ref) ** 2).sum() / (ref ** 2).sum())
        print(f"[gpu] relative RMS error {error:.1e}", flush=True)
        assert error <= tol
