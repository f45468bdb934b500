"""The largest owned cores of the order-5 build (12 x 12 x 20 = 2,880 points, at order 6
the limit is 2,208): 216 waters on 24 x 24 x 40 against the order-5 oracle, both
converged to 1e-10 Debye in the FP64 path (energy 1e-9, forces 1e-8 relative RMS,
the tolerances of the order-5 build's other tilings), 1e-6 Debye in the mixed path
(1e-6, 1e-5).  In a process of its own: the library and the oracle pick their
build at import.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECKS = """
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.waterbox import make_waterbox
from oracle import oracle
assert oracle.PME_ORDER == 5
force, pos, box = make_waterbox("water216", target_eps=1e-10)
force.setPMEParameters(force.getPMEParameters()[0], 24, 24, 40)
ref = oracle.evaluate(force.flatten(), pos, box)
for precision, eps, e_tol, f_tol in (("double", 1e-10, 1e-9, 1e-8), ("mixed", 1e-6, 1e-6, 1e-5)):
    force.setMutualInducedTargetEpsilon(eps)
    k = HipCalcMPIDForceKernel(precision, spread_tiling=(1, 1))
    k.initialize(len(pos), force, default_box=box)
    e, F = k.execute(pos, box)
    de = abs(e - ref["energy"]) / abs(ref["energy"])
    df = np.sqrt(((F - ref["forces"]) ** 2).sum() / (ref["forces"] ** 2).sum())
    print(precision, de, df, flush=True)
    assert de <= e_tol and df <= f_tol
"""


def test_order5_largest_cores():
    print("[gpu] order-5 build, cores of 2,880 points (subprocess)", flush=True)
    p = subprocess.run([sys.executable, "-u", "-c", CHECKS, ROOT], env=dict(os.environ, MPID_PME_ORDER="5"),
                       capture_output=True, text=True, timeout=100)
    print(p.stdout[-1000:], p.stderr[-1000:])
    assert p.returncode == 0, p.stdout + p.stderr
