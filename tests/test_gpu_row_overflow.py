"""A context reused at a density at which its block rows overflow.

After its first evaluation a context does not wait for the count of the block
rows: the list kernels run over the rows that fit, the count is read with the
solver's first check, and the evaluation is repeated with larger buffers.
30,000 atoms (a last block of 48) compressed by 0.85 per edge: the rows grow past
their capacity of 1.25 times the first count and 64.  The masks of every stored
row entry are read before the count is, so all of them have to be written (their
reads past the last atom would not show in the result).  The repeated evaluation
must give what a fresh context gives: the same kernels on the same inputs, so
the tolerances are those of the order of the sums on the grid, 1e-12 in energy and
1e-10 in forces in FP64, 1e-9 and 1e-6 in the mixed path.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import make_small_waterbox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,polarization",
                         [("double", MPIDForce.Mutual), ("mixed", MPIDForce.Mutual), ("mixed", MPIDForce.Direct),
                          ("mixed", MPIDForce.Extrapolated)],
                         ids=["double-mutual", "mixed-mutual", "mixed-direct", "mixed-extrapolated"])
def test_rows_overflow(precision, polarization):
    force, pos, box = make_small_waterbox(10000, 3, polarization=polarization)
    force.setPMEParameters(force.getPMEParameters()[0], 96, 96, 96)
    blocks = (len(pos) + 63) // 64
    k = HipCalcMPIDForceKernel(precision)
    k.initialize(len(pos), force, default_box=box)
    print(f"[gpu] row overflow, {precision}, polarization {polarization}", flush=True)
    k.execute(pos, box)
    rows = 2 * k.stats()["ntiles"] - blocks
    e1, f1 = k.execute(0.85 * pos, 0.85 * box)
    assert 2 * k.stats()["ntiles"] - blocks > rows + rows // 4 + 64  # the rows did overflow
    fresh = HipCalcMPIDForceKernel(precision)
    fresh.initialize(len(pos), force, default_box=box)
    e2, f2 = fresh.execute(0.85 * pos, 0.85 * box)
    tol_e, tol_f = (1e-12, 1e-10) if precision == "double" else (1e-9, 1e-6)
    assert abs(e1 - e2) <= tol_e * abs(e2)
    assert np.sqrt(((f1 - f2) ** 2).sum() / (f2 ** 2).sum()) <= tol_f
