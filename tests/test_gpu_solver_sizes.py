"""The evaluation's build and the mutual-polarization solver at the sizes where
their kernels change form.

Sorting and lab frames around whole 64-atom blocks and around 16,384 atoms (one
kernel ranks the keys and one workgroup builds the block rows up to there, a
radix sort and several kernels beyond): the lab-frame dipoles, which come back
through the permutation, equal the frames written out in numpy to 2e-13 of
the largest component (FP64 rounding: the O-H vectors carry 1e-15 of box edges
up to 5.5 nm, 6e-15 of the 0.0957 nm bond, through two normalisations and the
orthogonalisation, with a factor 10 in hand).

Small clusters without a cutoff, at site counts around the eight sites of an
operator workgroup, against the FP64 oracle converged to 1e-10 Debye: the
FP64 path at 1e-9 Debye within 1e-10 relative in energy (second order in the
residual) and 1e-7 relative RMS in forces (first order: 1e-9 Debye is about
1e-8 of the dipoles); the mixed path's forces within the workload bar of 1e-5
(a small cluster's energy is a difference of large pair terms that a relative
bar on the sum does not describe).

Extrapolated polarization with one to three coefficients (no order, one and two
orders) in a triclinic cell against the oracle: there is no iteration, so the
FP64 path differs by rounding and the fixed-point sums (1e-9 relative RMS in
forces and dipoles), the mixed path by the workload bar; and around 8,192 sites
the dipoles against the recursion written out with the inspection entry
points, to 1e-9 relative RMS (their fixed-point sums of 2^-32).

Periodic boxes around 2,048 sites (one workgroup updates all sites, beyond it
several do) and 8,192 sites (the operator's kernel adds the real-space field
itself, beyond it the list kernel does): the dipoles must satisfy the
equation they solve, mu = alpha (E0 + T mu), with E0 and T mu from the
inspection entry points, whose kernels are others.  The FP64 solve stops
below 1e-8 Debye RMS (over all atoms); E0 and T mu carry fixed-point sums of
2^-32, 1e-11 Debye at this alpha, so the residual formed from them must stay
below 1.01e-8 Debye.  The mixed path's dipoles agree with them to the
workload bar of 1e-5 relative RMS.
"""
import numpy as np
import pytest

from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import _o_parameters, _water_force, make_small_waterbox
from oracle import oracle

pytestmark = pytest.mark.gpu

DEBYE = 48.033324


def rel_rms(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum())


@pytest.mark.parametrize("waters", [1, 21, 22, 64, 65, 5461, 5462])
def test_lab_frames_through_the_sort(waters):
    force, pos, box = make_small_waterbox(max(waters, 32), waters)
    flat = force.flatten()
    k = HipCalcMPIDForceKernel("double")
    if waters < 32:  # a cluster: the smallest boxes hold 32 waters
        pos = pos[:3 * waters]
        force = _water_force(waters, _o_parameters(np.random.default_rng(waters), True, True))
        force.setNonbondedMethod(MPIDForce.NoCutoff)
        flat, box = force.flatten(), None
    k.initialize(len(pos), force, default_box=box)
    print(f"[gpu] frames of {waters} waters", flush=True)
    found = k.getLabFramePermanentDipoles(pos, box)
    o, h1, h2 = pos[0::3], pos[1::3], pos[2::3]

    def unit(v):
        return v / np.linalg.norm(v, axis=1, keepdims=True)

    u1, u2 = unit(h1 - o), unit(h2 - o)
    z = unit(u1 + u2)
    x = unit(u2 - z * (z * u2).sum(1, keepdims=True))
    d = flat["dipoles"].reshape(-1, 3)[0::3]
    expected = d[:, :1] * x + d[:, 1:2] * np.cross(z, x) + d[:, 2:] * z
    assert not found.reshape(-1, 3, 3)[:, 1:].any()
    assert np.abs(found[::3] - expected).max() <= 1e-14 * 20 * np.abs(expected).max()


@pytest.mark.parametrize("waters", [1, 2, 7, 8, 9, 33])
def test_small_clusters(waters):
    force, pos, _ = make_small_waterbox(waters, 40 + waters)
    force.setNonbondedMethod(MPIDForce.NoCutoff)
    force.setMutualInducedTargetEpsilon(1e-10)
    ref = oracle.evaluate(force.flatten(), pos, None)
    force.setMutualInducedTargetEpsilon(1e-9)
    for precision, e_tol, f_tol in (("double", 1e-10, 1e-7), ("mixed", None, 1e-5)):
        if precision == "mixed":
            force.setMutualInducedTargetEpsilon(1e-6)
        k = HipCalcMPIDForceKernel(precision)
        k.initialize(len(pos), force)
        print(f"[gpu] cluster of {waters} waters, {precision}", flush=True)
        e, F = k.execute(pos, None)
        # one molecule alone has no real-space pairs: its energy is zero
        if e_tol is not None:
            assert abs(e - ref["energy_variational"]) <= e_tol * max(abs(ref["energy_variational"]), 1.0)
        assert np.sqrt(((F - ref["forces"]) ** 2).sum()) <= f_tol * max(np.sqrt((ref["forces"] ** 2).sum()), 1.0)


@pytest.mark.parametrize("waters", [2048, 2049, 5461, 5462, 8192, 8193])
def test_dipoles_satisfy_their_equation(waters):
    alpha = 0.001
    rng = np.random.default_rng(waters)
    params = _o_parameters(rng, True, False)  # isotropic
    force, pos, box = make_small_waterbox(waters, waters, params)
    force.setMutualInducedTargetEpsilon(1e-8)
    k = HipCalcMPIDForceKernel("double")
    k.initialize(len(pos), force, default_box=box)
    print(f"[gpu] {waters} waters", flush=True)
    mu = k.getInducedDipoles(pos, box)
    st = k.stats()
    assert st["converged"] and st["epsilon"] < 1e-8
    assert not mu.reshape(-1, 3, 3)[:, 1:].any()  # hydrogens are not polarisable
    field = k.computeFixedField(pos, box) + k.computeInducedField(pos, box, mu)
    residual = (mu - alpha * field)[::3]
    assert DEBYE * np.sqrt((residual ** 2).sum() / len(pos)) <= 1.01e-8
    m = HipCalcMPIDForceKernel("mixed")
    force.setMutualInducedTargetEpsilon(1e-6)
    m.initialize(len(pos), force, default_box=box)
    assert rel_rms(m.getInducedDipoles(pos, box), mu) <= 1e-5


def test_no_polarisable_site():
    """Charges and multipoles only: nothing to solve, no iteration."""
    rng = np.random.default_rng(3)
    dip, quad, octo, _ = _o_parameters(rng, True, True)
    small, pos, box = make_small_waterbox(40, 3)
    force = _water_force(40, (dip, quad, octo, [0.0] * 3))
    force.setNonbondedMethod(MPIDForce.PME)
    force.setCutoffDistance(small.getCutoffDistance())
    force.setPMEParameters(*small.getPMEParameters())
    force.setPolarizationType(MPIDForce.Mutual)
    force.setMutualInducedTargetEpsilon(1e-6)
    ref = oracle.evaluate(force.flatten(), pos, box)
    for precision, e_tol, f_tol in (("double", 1e-9, 1e-9), ("mixed", 1e-6, 1e-5)):
        k = HipCalcMPIDForceKernel(precision)
        k.initialize(len(pos), force, default_box=box)
        print(f"[gpu] no polarisable site, {precision}", flush=True)
        e, F = k.execute(pos, box)
        assert k.stats()["iterations"] == 0
        assert abs(e - ref["energy"]) <= e_tol * abs(ref["energy"])
        assert rel_rms(F, ref["forces"]) <= f_tol


@pytest.mark.parametrize("coefficients", [[0.7], [0.3, 0.6], [-0.1, 0.4, 0.5]])
def test_extrapolation_orders(coefficients):
    force, pos, box = make_small_waterbox(60, 5, polarization=MPIDForce.Extrapolated)
    force.setExtrapolationCoefficients(coefficients)
    cutoff = 0.42
    force.setCutoffDistance(cutoff)
    force.setPMEParameters(2.628 / cutoff, 18, 20, 24)
    L = box[0]
    cell = np.array([[L, 0, 0], [0.2 * L, L, 0], [-0.15 * L, 0.1 * L, L]])
    ref = oracle.evaluate(force.flatten(), pos, cell, details=True)
    for precision, tol in (("double", 1e-9), ("mixed", 1e-5)):
        k = HipCalcMPIDForceKernel(precision)
        k.initialize(len(pos), force, default_box=cell)
        print(f"[gpu] {len(coefficients)} extrapolation coefficients, {precision}", flush=True)
        e, F = k.execute(pos, cell)
        assert rel_rms(F, ref["forces"]) <= tol
        assert rel_rms(k.getInducedDipoles(pos, cell), ref["induced"]) <= tol


@pytest.mark.parametrize("waters", [8192, 8193])
def test_extrapolation_recursion(waters):
    alpha = 0.001
    params = _o_parameters(np.random.default_rng(waters), True, False)  # isotropic
    force, pos, box = make_small_waterbox(waters, waters, params, polarization=MPIDForce.Extrapolated)
    coefficients = [0.2, 0.3, 0.5]
    force.setExtrapolationCoefficients(coefficients)
    k = HipCalcMPIDForceKernel("double")
    k.initialize(len(pos), force, default_box=box)
    print(f"[gpu] {waters} waters, extrapolated", flush=True)
    found = k.getInducedDipoles(pos, box)
    site = np.zeros((len(pos), 1))
    site[::3] = alpha
    order = site * k.computeFixedField(pos, box)
    expected = sum(coefficients) * order
    for m in (1, 2):
        order = site * k.computeInducedField(pos, box, order)
        expected = expected + sum(coefficients[m:]) * order
    assert rel_rms(found, expected) <= 1e-9


@pytest.mark.parametrize("polarization", [MPIDForce.Mutual, MPIDForce.Direct, MPIDForce.Extrapolated],
                         ids=["mutual", "direct", "extrapolated"])
def test_repeated_evaluations_without_cutoff(polarization):
    force, pos, _ = make_small_waterbox(216, 5, polarization=polarization)
    force.setNonbondedMethod(MPIDForce.NoCutoff)
    force.setMutualInducedTargetEpsilon(1e-9)
    k = HipCalcMPIDForceKernel("double")
    k.initialize(len(pos), force)
    print(f"[gpu] repeated evaluations, polarization {polarization}", flush=True)
    first = k.execute(pos, None)[1]
    for _ in range(6):
        assert rel_rms(k.execute(pos, None)[1], first) <= 1e-12
