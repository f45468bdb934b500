"""PME grids over every split of the transforms' register steps: each axis takes
a different size per case, among them ones without a split (75, 125 as
either axis of a plane) and planes that exceed the LDS of a workgroup.

A box of 32 waters against the FP64 oracle on the same grid, converged to 1e-10
Debye.  The FP64 path at 1e-9 Debye: forces within 1e-7 relative RMS (first order
in the residual, 1e-8 of the dipoles; transforms and fixed-point sums are at
1e-13).  The mixed path, on grids of at most 64: 1e-5, the bar of the workloads.
(On finer ones, 0.01 nm here, FP32 spline derivatives in units of the spacing
limit it: 4e-5 whatever the transform.)
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.waterbox import make_small_waterbox
from oracle import oracle

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum())


@pytest.mark.parametrize("grid", [(12, 15, 16), (18, 20, 24), (25, 27, 30), (32, 36, 40), (45, 48, 50), (54, 60, 64),
                                  (72, 80, 81), (90, 96, 100), (100, 60, 12), (108, 40, 18), (40, 75, 20),
                                  (125, 24, 15), (120, 128, 16), (144, 20, 27), (20, 144, 128)])
def test_grid(grid):
    force, pos, box = make_small_waterbox(32, 21)
    force.setPMEParameters(force.getPMEParameters()[0], *grid)
    force.setMutualInducedTargetEpsilon(1e-10)
    ref = oracle.evaluate(force.flatten(), pos, box)["forces"]
    for precision, eps, tol in (("double", 1e-9, 1e-7), ("mixed", 1e-6, 1e-5)):
        if precision == "mixed" and max(grid) > 64:
            continue
        force.setMutualInducedTargetEpsilon(eps)
        k = HipCalcMPIDForceKernel(precision)
        k.initialize(len(pos), force, default_box=box)
        print(f"[gpu] grid {grid} {precision}", flush=True)
        assert rel_rms(k.execute(pos, box)[1], ref) <= tol
