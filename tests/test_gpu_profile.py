"""Profiled kernel families: the covalent pairs' electrostatics, a part of the
per-atom dispatch otherwise, are timed apart when their family is asked for, once
per evaluation, and the forces do not change by it (integer sums: what differs
is the order of the FP64 sums on the grid, 1e-10 relative RMS).
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import make_small_waterbox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("polarization", [MPIDForce.Mutual, MPIDForce.Direct, MPIDForce.Extrapolated],
                         ids=["mutual", "direct", "extrapolated"])
def test_covalent_pairs_are_timed(polarization):
    force, pos, box = make_small_waterbox(100, 9, polarization=polarization, target_eps=1e-9)
    k = HipCalcMPIDForceKernel("double")
    k.initialize(len(pos), force, default_box=box)
    print(f"[gpu] covalent pairs profiled, polarization {polarization}", flush=True)
    plain = k.execute(pos, box)[1]
    for families in (["covalent_pairs"], ["covalent_pairs", "recip_atoms"]):
        k.setProfileFamilies(families)
        k.profile(reset=True)
        for _ in range(3):
            timed = k.execute(pos, box)[1]
        profile = k.profile(reset=True)
        for name in families:
            assert profile[name][1] == 3 and profile[name][0] > 0.0, name
        assert np.sqrt(((timed - plain) ** 2).sum() / (plain ** 2).sum()) <= 1e-10
    k.setProfileFamilies(["recip_atoms"])
    k.execute(pos, box)
    assert k.profile(reset=True)["covalent_pairs"][1] == 0
