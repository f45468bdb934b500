"""The block rows where their kernels change form: up to 64 blocks (4,096 atoms) one
workgroup counts, scans and writes them, beyond that three dispatches do.

Boxes of 4,095 atoms (64 blocks, all of that workgroup's rows) and 4,098 atoms
(65 blocks, the last of two atoms) with direct polarization against the FP64
oracle: there is no iteration, so the FP64 path differs by rounding and the
fixed-point sums (1e-9 relative RMS), the mixed path by the workload bar (1e-5).
A missing or doubled row changes the forces of a whole block.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import make_small_waterbox
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters", [1365, 1366])
def test_block_rows(waters):
    force, pos, box = make_small_waterbox(waters, waters, polarization=MPIDForce.Direct)
    ref = oracle.evaluate(force.flatten(), pos, box)["forces"]
    for precision, tol in (("double", 1e-9), ("mixed", 1e-5)):
        k = HipCalcMPIDForceKernel(precision)
        k.initialize(len(pos), force, default_box=box)
        print(f"[gpu] {waters} waters, {precision}", flush=True)
        for _ in range(2):  # the second time the rows are not waited for
            F = k.execute(pos, box)[1]
            assert np.sqrt(((F - ref) ** 2).sum() / (ref ** 2).sum()) <= tol
