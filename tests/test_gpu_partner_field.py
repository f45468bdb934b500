"""A covalent partner's induced field beside a much larger one of the listed
neighbours, mixed precision.

Extrapolated polarization without a cutoff, two coefficients: the dipole of site
0 is c'_0 mu_0 + c'_1 alpha E_1, E_1 the field of the first dipoles.  Its covalent
partner, site 1, carries no moments and a polarisability of 1e-13 nm^3, so that
its share of E_1 is about 1e-9 of the neighbours': less than half a unit of their
FP32 sum.  Doubling that polarisability changes nothing else, bit for bit; the
difference of the two dipoles must be the partner's field as the FP64 path gives
it.  FP32 holds that field to a few 1e-7 (its factors' roundings), the
difference of two FP64 dipoles to 1e-6: within 1e-4.  (Added to the neighbours in
FP32, the field is lost: a relative error of 1.)  With 4 polarisable sites one
kernel does all of an order; with 8,200 the lists have their own.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce

pytestmark = pytest.mark.gpu


def dipole_of_first(precision, n, alpha):
    pos = [(0.0, 0.0, 0.0), (0.06, 0.05, 0.07), (0.25, -0.1, 0.15), (-0.2, 0.24, 0.1)]
    charge = [0.3, 0.0, -0.5, 0.4]
    pos += [(2.0 + 0.5 * (a % 20), 2.0 + 0.5 * (a // 20 % 20), 2.0 + 0.5 * (a // 400)) for a in range(n - 4)]
    force = MPIDForce()
    for a in range(n):
        polarity = [alpha if a == 1 else 0.001] * 3
        force.addMultipole(charge[a] if a < 4 else 0.0, [0.0] * 3, [0.0] * 6, [0.0] * 10, MPIDForce.NoAxisType, -1, -1,
                           -1, 1.3, polarity)
    force.setCovalentMap(0, MPIDForce.Covalent12, [1])
    force.setCovalentMap(1, MPIDForce.Covalent12, [0])
    force.setDefaultTholeWidth(5.0)
    force.setNonbondedMethod(MPIDForce.NoCutoff)
    force.setPolarizationType(MPIDForce.Extrapolated)
    force.setExtrapolationCoefficients([0.4, 0.6])
    k = HipCalcMPIDForceKernel(precision)
    k.initialize(n, force)
    return k.getInducedDipoles(np.array(pos), None)[0]


@pytest.mark.parametrize("n", [4, 8200])
def test_small_field_of_a_partner_is_kept(n):
    change = {}
    for precision in ("double", "mixed"):
        print(f"[gpu] partner field, {n} sites, {precision}", flush=True)
        change[precision] = dipole_of_first(precision, n, 2e-13) - dipole_of_first(precision, n, 1e-13)
    error = np.sqrt(((change["mixed"] - change["double"]) ** 2).sum() / (change["double"] ** 2).sum())
    print(f"[gpu] change {change['double']}, relative error {error:.1e}", flush=True)
    assert error <= 1e-4
