"""Host-buffer evaluations (staged through pinned memory up to 16,384 atoms, by
copies beyond) against the device-buffer entry point, forces added to the
caller's, twice through the same buffers; and the dipoles that follow against
those of a context of their own.  The kernels are the same; what may differ is
the order of the FP32 sums on the grid (and of the solver's steps on them): 2^-24
each, 1e-6 relative RMS with a factor sixteen in hand.
"""
import numpy as np
import pytest
import torch

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.waterbox import make_small_waterbox

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum())


@pytest.mark.parametrize("waters", [32, 5461, 5462])
def test_host_and_device_buffers_agree(waters):
    force, pos, box = make_small_waterbox(waters, 17)
    k = HipCalcMPIDForceKernel("mixed")
    k.initialize(len(pos), force, default_box=box)
    print(f"[gpu] host buffers, {3 * waters} atoms", flush=True)
    start = np.random.default_rng(1).normal(0.0, 100.0, size=pos.shape)
    d_pos = torch.tensor(pos, dtype=torch.float64, device="cuda")
    for shift in (0.0, 0.01):  # a second, different configuration through the same buffers
        p = pos + shift * np.sin(np.arange(pos.size)).reshape(pos.shape) * 0.1
        d_pos.copy_(torch.from_numpy(p))
        d_forces = torch.tensor(start, device="cuda")
        torch.cuda.synchronize()
        e_dev = k.execute_device(d_pos.data_ptr(), box, d_forces.data_ptr())
        torch.cuda.synchronize()
        mine = start.copy()
        e, f = k.execute(p, box, forces=mine)
        dipoles = k.getInducedDipoles(p, box)
        only = k.execute(p, box, includeForces=False)[0]
        assert abs(e - e_dev) <= 1e-6 * abs(e_dev) and abs(only - e_dev) <= 1e-6 * abs(e_dev)
        assert rel_rms(f - start, d_forces.cpu().numpy() - start) <= 1e-6
        fresh = HipCalcMPIDForceKernel("mixed")
        fresh.initialize(len(pos), force, default_box=box)
        assert rel_rms(dipoles, fresh.getInducedDipoles(p, box)) <= 1e-6
