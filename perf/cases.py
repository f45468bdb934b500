"""Performance cases of the MPIDForce evaluator: what programs that use it have it do.

Kinds of cases:

step       one energy + force evaluation of a molecular-dynamics or scoring
           program.  Device buffers (``execute_device``: positions and forces
           stay in GPU memory, the program clears the force buffer before each
           step, as an MD engine does) or host buffers (``execute`` on numpy
           arrays, as a script around ``MPIDContext`` does), optionally
           followed by the induced dipoles of the same configuration.
gradients  one step of a parameter fit: the energy of a box through
           ``MPIDEnergy`` with float32 parameter leaves, and its gradients
           with respect to every per-particle parameter.
batch      a score of many independent small boxes through ``BatchEvaluator``.

All systems are boxes of water (O: charge, dipole, quadrupole, octopole,
polarisability; H: charge) on a jittered lattice at liquid density, drawn from
the seed: the workloads of ``mpidopenmmplugin_amd.waterbox`` (216, 4,096 and
32,768 waters, the 512-system batch) and boxes of other shapes with lattice
sites left empty, so that atom counts are ragged and PME grids odd or
different along each axis.

Programs in mixed precision keep forces, dipoles and gradients in float32
(their accuracy is a few 1e-6); programs in double precision keep float64.
"""
import math

import numpy as np
import torch

from mpidopenmmplugin_amd.autograd import PARAMETERS, MPIDEnergy
from mpidopenmmplugin_amd.batch import BatchEvaluator
from mpidopenmmplugin_amd.kernel import HipCalcMPIDForceKernel
from mpidopenmmplugin_amd.mpidforce import MPIDForce
from mpidopenmmplugin_amd.waterbox import (_o_parameters, _water_force, _waters, ewald_alpha, make_small_waterbox,
                                           smooth_235)

SPACING = 0.310375  # nm between lattice sites: 32 of them make the 9.932 nm box
POLARIZATION = {"mutual": MPIDForce.Mutual, "direct": MPIDForce.Direct, "extrapolated": MPIDForce.Extrapolated}


def _box_case(name, kx, ky, kz, waters=None, **more):
    case = dict(kind="step", kx=kx, ky=ky, kz=kz, waters=kx * ky * kz if waters is None else waters, method="pme",
                polarization="mutual", precision="mixed", anisotropic=True, buffers="device", dipoles=False)
    if name:
        case["name"] = name
    case.update(more)
    if case["method"] == "pme":
        short = SPACING * min(kx, ky, kz)
        case.setdefault("cutoff", min(0.8, round(0.5 * short - 1e-3, 6)))
        for axis, k in zip("xyz", (kx, ky, kz)):
            case.setdefault("g" + axis, max(6, smooth_235(math.ceil(SPACING * k / 0.08))))
    return case


def listed():
    return [
        # gas-phase cluster of a conformer or many-body scan: no cutoff, no grid, the smallest call
        _box_case("cluster_27_double", 3, 3, 3, method="nocutoff", precision="double", buffers="host"),
        # the smallest periodic box of the batched workload, evaluated on its own: launches and latency only
        _box_case("pme_32_mixed", 4, 3, 3, waters=32, buffers="host"),
        # the 648-atom box of the reference's water tests, energy, forces and induced dipoles to a script
        _box_case("pme_216_dipoles_mixed", 6, 6, 6, gx=24, gy=24, gz=24, anisotropic=False, buffers="host",
                  dipoles=True),
        # an MD step of an ordinary small box with the force-field generator's default polarization
        _box_case("md_996_extrapolated_mixed", 10, 10, 10, waters=996, polarization="extrapolated"),
        # an MD step of the 12,288-atom box, in both precisions
        _box_case("md_4096_mixed", 16, 16, 16, gx=64, gy=64, gz=64),
        _box_case("md_4096_double", 16, 16, 16, gx=64, gy=64, gz=64, precision="double"),
        # one step of a parameter fit on the same box
        _box_case("gradients_4096_mixed", 16, 16, 16, gx=64, gy=64, gz=64, kind="gradients"),
        # an elongated box with a ragged atom count (direct polarization, a different grid along z)
        _box_case("md_slab_9973_direct_mixed", 20, 20, 25, waters=9973, polarization="direct"),
        # the 98,304-atom box: the headline MD step, its double-precision form, and the generator's default
        _box_case("md_32768_mixed", 32, 32, 32, gx=128, gy=128, gz=128, cutoff=0.9),
        _box_case("md_32768_double", 32, 32, 32, gx=128, gy=128, gz=128, cutoff=0.9, precision="double"),
        _box_case("md_32768_extrapolated_mixed", 32, 32, 32, gx=128, gy=128, gz=128, cutoff=0.9,
                  polarization="extrapolated"),
        # scoring of many small boxes of 32-1024 waters at once
        dict(name="batch_64_mixed", kind="batch", systems=64, lo=32, hi=1024, precision="mixed"),
    ]


def draw(rng):
    """One more case of the same ranges: boxes of 27 to 32,768 sites (cubic to twice as long as wide, some sites
    empty), clusters of up to 343 waters, fits of up to 4,096 waters, batches of 8 to 48 systems."""
    kind = rng.choice(["host", "device", "device", "device", "cluster", "gradients", "batch"])
    precision = rng.choice(["mixed", "mixed", "double"])
    polarization = rng.choice(["mutual", "mutual", "direct", "extrapolated"])
    if kind == "batch":
        lo = rng.randint(32, 128)
        return dict(kind="batch", systems=rng.randint(8, 48), lo=lo, hi=rng.randint(2 * lo, 1024),
                    precision=precision)
    low, high = {"host": (36, 1000), "device": (300, 32768), "cluster": (27, 343), "gradients": (64, 4096)}[kind]
    sites = math.exp(rng.uniform(math.log(low), math.log(high)))
    aspect = rng.uniform(1.0, 2.0)
    k = (sites / aspect) ** (1.0 / 3.0)
    kx, ky, kz = max(3, int(k)), max(3, int(round(k))), max(3, int(k * aspect))
    while kx * ky * kz > high:
        kz -= 1
    waters = kx * ky * kz - rng.randint(0, max(1, kx * ky * kz // 25))
    more = dict(precision=precision, polarization=polarization, anisotropic=rng.random() < 0.7)
    if kind == "cluster":
        more.update(method="nocutoff", buffers="host")
    elif kind == "host":
        more.update(buffers="host", dipoles=rng.random() < 0.5)
    elif kind == "gradients":
        more.update(kind="gradients", polarization=rng.choice(["mutual", "mutual", "direct"]), precision="mixed")
    elif min(kx, ky, kz) >= 6 and rng.random() < 0.3:
        more.update(cutoff=0.9)
    return _box_case(None, kx, ky, kz, waters=waters, **more)


def _system(case, seed):
    """(force, positions [n,3], box edges [3]) of a box case."""
    rng = np.random.default_rng([int(seed), 20261205])
    params = _o_parameters(rng, True, case["anisotropic"])
    kx, ky, kz = case["kx"], case["ky"], case["kz"]
    sites = np.stack(np.meshgrid(np.arange(kx), np.arange(ky), np.arange(kz), indexing="ij"), -1).reshape(-1, 3)
    sites = sites[np.sort(rng.choice(len(sites), size=case["waters"], replace=False))]
    pos = _waters(rng, sites.astype(np.float64), SPACING)
    force = _water_force(case["waters"], params)
    force.setPolarizationType(POLARIZATION[case["polarization"]])
    force.setMutualInducedTargetEpsilon(1e-6)
    if case["method"] == "nocutoff":
        force.setNonbondedMethod(MPIDForce.NoCutoff)
        return force, pos, None
    force.setNonbondedMethod(MPIDForce.PME)
    force.setCutoffDistance(case["cutoff"])
    force.setPMEParameters(ewald_alpha(case["cutoff"]), case["gx"], case["gy"], case["gz"])
    return force, pos, SPACING * np.array([kx, ky, kz], dtype=np.float64)


def _rows(values, n):
    """Flat per-particle values as MPIDEnergy takes them: [n], or a row of components for each particle."""
    return values if values.shape[0] == n else values.reshape(n, -1)


def _batch_systems(case, seed):
    rng = np.random.default_rng([int(seed), 20261206])
    params = _o_parameters(rng, True, True)
    # the same systems' sizes for every seed: the user's set of molecules stays, their configurations change
    sizes = np.random.default_rng([case["systems"], case["lo"]]).integers(case["lo"], case["hi"] + 1, case["systems"])
    return [make_small_waterbox(int(m), [int(seed), i], params) for i, m in enumerate(sizes)]


def prepare(case, seed):
    state = dict(case=case, keep=np.float32 if case["precision"] == "mixed" else np.float64)
    if case["kind"] == "batch":
        state["batch"] = BatchEvaluator(_batch_systems(case, seed), precision=case["precision"])
        return state
    force, pos, box = _system(case, seed)
    state["box"] = box
    if case["kind"] == "gradients":
        flat = force.flatten()
        state["model"] = MPIDEnergy(force, box, precision=case["precision"])
        state["positions"] = torch.from_numpy(pos)
        state["leaves"] = [torch.tensor(_rows(flat[k], len(pos)), dtype=torch.float32).requires_grad_(True)
                           for k in PARAMETERS]
        state["leaves"].append(torch.tensor(flat["default_thole"], dtype=torch.float32).requires_grad_(True))
        return state
    kernel = HipCalcMPIDForceKernel(case["precision"])
    kernel.initialize(len(pos), force, default_box=box)
    state["kernel"] = kernel
    if case["buffers"] == "device":
        state["positions"] = torch.from_numpy(pos).cuda()
        state["forces"] = torch.zeros(len(pos), 3, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
    else:
        state["positions"] = pos
    return state


def run(state):
    case, keep = state["case"], state["keep"]
    if case["kind"] == "batch":
        energies, forces = zip(*state["batch"].execute())
        return dict(energies=np.array(energies, dtype=keep),
                    forces=np.concatenate(forces, dtype=keep, casting="same_kind"))
    if case["kind"] == "gradients":
        energy = state["model"](state["positions"], *state["leaves"])
        return dict(energy=energy.item(), **dict(zip(PARAMETERS + ("default_thole",),
                                                     torch.autograd.grad(energy, state["leaves"]))))
    kernel = state["kernel"]
    if case["buffers"] == "device":
        forces = state["forces"].zero_()
        torch.cuda.current_stream().synchronize()  # the evaluator works on streams of its own
        energy = kernel.execute_device(state["positions"].data_ptr(), state["box"], forces.data_ptr())
        return dict(energy=energy, forces=forces.float() if keep is np.float32 else forces)
    energy, forces = kernel.execute(state["positions"], state["box"])
    out = dict(energy=energy, forces=forces.astype(keep, copy=False))
    if case["dipoles"]:
        out["dipoles"] = kernel.getInducedDipoles(state["positions"], state["box"]).astype(keep, copy=False)
    return out


def _box_work(waters, volume, cutoff, grid, polarization, gradients, precision):
    """Bytes and operations of one evaluation: the atoms' inputs and outputs once; the pairs within the cutoff once in
    the field and the energy kernels and, for polarisable pairs, in each solver product; the grid products of one
    permanent and one induced cycle per product (6 x 6 x 6 points an atom, 5 n log2 n per transform)."""
    n = 3 * waters
    pairs = n * (n - 1) / 2 if not grid else 0.5 * n * n / volume * 4.0 / 3.0 * math.pi * cutoff ** 3
    pol, one, bare = pairs / 9, 4 * pairs / 9, 4 * pairs / 9
    products = {"mutual": 8, "direct": 1, "extrapolated": 3}[polarization] + (4 if gradients else 0)
    flops = pol * (2106 + 283 + 66 * products) + one * (568 + 152) + bare * 19
    if grid:
        points = grid[0] * grid[1] * grid[2]
        cycle = 2 * 2.5 * points * math.log2(points) + points
        flops += (products + 1) * cycle + 216 * n * (2 * 20 + 2 * 35) + products * 216 * waters * (2 * 3 + 2 * 3)
    # positions, forces (added: read and written), charges and frames of all; 20 moments and polarisabilities of O
    nbytes = n * (24 + 48 + 8 + 16 + 16) + waters * (20 * 8 + 6 * 8)
    if gradients:
        nbytes = n * (24 + 2 * 24 * 4)
    return nbytes, flops


def work(case):
    if case["kind"] == "batch":
        mean = 0.5 * (case["lo"] + case["hi"])
        edge = (mean / 33.428) ** (1.0 / 3.0)
        b, f = _box_work(mean, edge ** 3, min(0.8, 0.5 * edge), [edge / 0.08] * 3, "mutual", False, "mixed")
        return dict(bytes=b * case["systems"], flops=f * case["systems"])
    grid = [case["gx"], case["gy"], case["gz"]] if case["method"] == "pme" else None
    b, f = _box_work(case["waters"], case["kx"] * case["ky"] * case["kz"] * SPACING ** 3, case.get("cutoff"), grid,
                     case["polarization"], case["kind"] == "gradients", case["precision"])
    return dict(bytes=b, flops=f)


# ---- the same quantities in plain float64 torch ---------------------------------------
# The energy is written down once as a function of positions, moments, dipoles and damping, from Ewald's split of the
# Coulomb sum, Thole's damping and cardinal B-splines of order 6; forces and gradients are its automatic derivatives
# at the converged dipoles.
COULOMB = 138.935455846
SQRT_PI = 1.77245385091
POWERS = [(a, b, c) for total in range(7) for a in range(total, -1, -1) for b in range(total - a, -1, -1)
          for c in [total - a - b]]
PLACE = {p: i for i, p in enumerate(POWERS)}
WEIGHT = [math.factorial(sum(p)) / (math.factorial(p[0]) * math.factorial(p[1]) * math.factorial(p[2]))
          for p in POWERS[:20]]
PAIR = [[PLACE[tuple(x + y for x, y in zip(p, q))] for q in POWERS[:20]] for p in POWERS[:20]]
SIGN = [(-1.0) ** sum(p) for p in POWERS[:20]]
TENSOR2 = [[PLACE[tuple((i == k) + (j == k) for k in range(3))] - 4 for j in range(3)] for i in range(3)]
TENSOR3 = [[[PLACE[tuple((i == k) + (j == k) + (m == k) for k in range(3))] - 10 for m in range(3)] for j in range(3)]
           for i in range(3)]
CHUNK = 100000  # pairs held at once


def _radial(r, alpha, top):
    """Ewald's B_0..B_top and the bare (2k-1)!!/r^(2k+1)."""
    ex = torch.exp(-(alpha * r) ** 2)
    screened, bare = [torch.erfc(alpha * r) / r], [1.0 / r]
    for k in range(1, top + 1):
        gauss = (2 * alpha * alpha) ** k / (alpha * SQRT_PI) * ex if alpha else 0.0
        screened.append(((2 * k - 1) * screened[-1] + gauss) / r ** 2)
        bare.append((2 * k - 1) * bare[-1] / r ** 2)
    return screened, bare


def _thole(u):
    """The damping factors of the bare terms of order 3, 5, 7 and 9 (the first entry, of the charge term, is 1)."""
    e = torch.exp(-u)
    p3 = 1 + u + u ** 2 / 2
    p5 = p3 + u ** 3 / 6
    return [torch.ones_like(u), 1 - e * p3, 1 - e * p5, 1 - e * (p5 + u ** 4 / 30),
            1 - e * (p5 + 4 * u ** 4 / 105 + u ** 5 / 210)]


def _tensor(d, g):
    """All Cartesian derivatives of the radial function with (1/r d/dr)^k f = (-1)^k g_k, one column for each power up
    to the order of g, by the recursion over the powers."""
    top = len(g) - 1
    level = {(0, 0, 0): [(-1.0) ** k * g[k] for k in range(top + 1)]}
    for p in POWERS[1:]:
        if sum(p) > top:
            break
        axis = next(k for k in range(3) if p[k])
        low = tuple(p[k] - (k == axis) for k in range(3))
        lower = tuple(p[k] - 2 * (k == axis) for k in range(3))
        level[p] = [d[:, axis] * level[low][k + 1] + (low[axis] * level[lower][k + 1] if low[axis] else 0.0)
                    for k in range(top + 1 - sum(p))]
    return torch.stack([level[p][0] for p in POWERS if sum(p) <= top], 1)


def _frames(pos, flat):
    """Rows: the molecular x, y and z axes (bisector sites and z-then-x sites)."""
    unit = lambda v: v / v.norm(dim=1, keepdim=True)  # noqa: E731
    index = lambda k: torch.as_tensor(flat[k], dtype=torch.long, device=pos.device)  # noqa: E731
    z, x = unit(pos[index("atom_z")] - pos), unit(pos[index("atom_x")] - pos)
    bisector = (index("axis_types") == MPIDForce.Bisector)[:, None]
    z = unit(torch.where(bisector, z + x, z))
    x = unit(x - z * (z * x).sum(1, keepdim=True))
    return torch.stack([x, torch.linalg.cross(z, x), z], 1)


def _moments(axes, charges, dipoles, quadrupoles, octopoles):
    """The 20 lab-frame moments, each with the number of index orders that it stands for.  Inputs in the order of
    MPIDForce: XX XY YY XZ YZ ZZ; XXX XXY XYY YYY XXZ XYZ YYZ XZZ YZZ ZZZ."""
    n = len(charges)
    quad = quadrupoles.reshape(n, 6)[:, [0, 1, 3, 2, 4, 5]]
    octo = octopoles.reshape(n, 10)[:, [0, 1, 4, 2, 5, 7, 3, 6, 8, 9]]
    q = torch.einsum("nij,nia,njb->nab", quad[:, TENSOR2], axes, axes)
    o = torch.einsum("nijk,nia,njb,nkc->nabc", octo[:, TENSOR3], axes, axes, axes)
    d = torch.einsum("ni,nia->na", dipoles.reshape(n, 3), axes)
    flat = [charges] + [d[:, i] for i in range(3)]
    flat += [q[:, i, j] for i in range(3) for j in range(i, 3)]
    flat += [o[:, i, j, k] for i in range(3) for j in range(i, 3) for k in range(j, 3)]
    return torch.stack(flat, 1) * torch.tensor(WEIGHT, dtype=torch.float64, device=axes.device)


def _pairs(pos, box, cutoff):
    n, out = len(pos), []
    rows = max(1, int(2e7) // n)
    for a in range(0, n, rows):
        near = torch.ones(min(rows, n - a), n - a, dtype=torch.bool, device=pos.device).triu(1)
        if box is not None:
            r2 = torch.zeros(near.shape, dtype=torch.float64, device=pos.device)
            for k in range(3):
                x = pos[a:a + rows, k:k + 1] - pos[None, a:, k]
                r2 += (x - box[k] * torch.floor(x / box[k] + 0.5)) ** 2
            near &= r2 <= cutoff ** 2
        out.append(near.nonzero() + a)
    return torch.cat(out)


def _splines(fraction):
    """Order-6 cardinal B-spline weights of the 6 grid points and their derivatives up to the third: [n, 4, 6]."""
    pad = torch.nn.functional.pad
    m = torch.arange(7, dtype=torch.float64, device=fraction.device)
    w, table = fraction[:, None], {}
    c = torch.ones_like(w)
    for p in range(1, 7):
        if p > 1:
            left, right = pad(c, (1, 0)), pad(c, (0, 1))
            c = ((w + (p - 1 - m[:p])) * left + (m[:p] + 1 - w) * right) / (p - 1)
        table[p] = c
    out = [table[6]]
    for r in range(1, 4):
        c = table[6 - r]
        for _ in range(r):
            c = pad(c, (1, 0)) - pad(c, (0, 1))
        out.append(c)
    return torch.stack(out, 1)


class _Mesh:
    """The reciprocal-space sum on the grid of the case."""

    def __init__(self, box, grid, alpha, device):
        self.box, self.grid, self.alpha, self.device = box, grid, alpha, device
        m, moduli = [], []
        for k in range(3):
            index = np.arange(grid[k])
            m.append(np.where(index < (grid[k] + 1) // 2, index, index - grid[k]) / box[k])
            moduli.append(self._moduli(grid[k]))
        m2 = m[0][:, None, None] ** 2 + m[1][:, None] ** 2 + m[2] ** 2
        m2[0, 0, 0] = 1.0
        g = np.exp(-math.pi ** 2 * m2 / alpha ** 2) / (math.pi * np.prod(box) * m2)
        g /= moduli[0][:, None, None] * moduli[1][:, None] * moduli[2]
        g[0, 0, 0] = 0.0
        self.influence = torch.from_numpy(g).to(device)

    @staticmethod
    def _moduli(n):
        """|b(m)|^2 of the order-6 spline with the aliasing sums' least-squares factor (100 images)."""
        weights = _splines(torch.zeros(1, dtype=torch.float64))[0, 0].numpy()
        b = np.abs(np.exp(2j * math.pi * np.outer(np.arange(n), np.arange(1, 7)) / n) @ weights) ** 2
        index = np.arange(n)
        k = np.where(index + 1 > n // 2, index - n, index).astype(np.float64)
        k[0] = 0.0
        f = math.pi * k[:, None] / n
        j = math.pi * np.concatenate([np.arange(1, 51), -np.arange(1, 51)])
        ratio = f / (f + j)
        zeta = (1 + (ratio ** 12).sum(1)) / (1 + (ratio ** 6).sum(1))
        return b * zeta ** 2

    def _stencil(self, pos):
        theta, cells = [], []
        for k in range(3):
            x = pos[:, k] / self.box[k]
            x = (x - torch.floor(x + 0.5) + 0.5) * self.grid[k]
            start = torch.floor(x.detach())
            cells.append((start.long()[:, None] - 5 + torch.arange(6, device=self.device)) % self.grid[k])
            scale = torch.tensor([(self.grid[k] / self.box[k]) ** r for r in range(4)], dtype=torch.float64,
                                 device=self.device)
            theta.append(_splines(x - start) * scale[:, None])
        place = (cells[0][:, :, None, None] * self.grid[1] + cells[1][:, None, :, None]) * self.grid[2]
        return theta, place + cells[2][:, None, None, :]

    def potential(self, pos, moments):
        """The potential grid of the moments."""
        rho = torch.zeros(self.grid[0] * self.grid[1] * self.grid[2], dtype=torch.float64, device=self.device)
        for a in range(0, len(pos), 32768):
            (tx, ty, tz), place = self._stencil(pos[a:a + 32768])
            cube = torch.zeros(len(tx), 4, 4, 4, dtype=torch.float64, device=self.device)
            for k, (i, j, m) in enumerate(POWERS[:20]):
                cube[:, i, j, m] = moments[a:a + 32768, k]
            value = torch.einsum("nijm,nix->nxjm", cube, tx)
            value = torch.einsum("nxjm,njy->nxym", value, ty)
            rho.index_add_(0, place.reshape(-1), torch.einsum("nxym,nmz->nxyz", value, tz).reshape(-1))
        spectrum = torch.fft.fftn(rho.reshape(self.grid)) * self.influence
        return torch.fft.ifftn(spectrum).real.reshape(-1) * rho.numel()

    def derivatives(self, pos, potential):
        """The 20 derivatives of a potential grid at the atoms, differentiable in the positions."""
        (tx, ty, tz), place = self._stencil(pos)
        value = torch.einsum("nxyz,nmz->nxym", potential[place], tz)
        value = torch.einsum("nxym,njy->nxjm", value, ty)
        value = torch.einsum("nxjm,nix->nijm", value, tx)
        return torch.stack([value[:, i, j, m] for i, j, m in POWERS[:20]], 1)


class _Exact:
    """Energy, forces, induced dipoles and parameter gradients of one box."""

    def __init__(self, force, pos, box):
        self.device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        as64 = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.float64, device=self.device)  # noqa: E731
        self.flat, self.box = force.flatten(), None if box is None else as64(box)
        self.alpha = self.flat["alpha"] if box is not None else 0.0
        self.mesh = _Mesh(box, list(self.flat["grid"]), self.alpha, self.device) if box is not None else None
        self.pos = as64(pos).requires_grad_(True)
        self.leaves = [as64(self.flat[k]).requires_grad_(True) for k in PARAMETERS]
        self.leaves.append(as64(self.flat["default_thole"]).requires_grad_(True))
        polarity = self.flat["polarity"].reshape(len(pos), 3)
        self.polar = torch.as_tensor(polarity.sum(1) > 0, device=self.device)
        self.sites = self.polar.nonzero()[:, 0]
        with torch.no_grad():
            pairs = _pairs(self.pos, self.box, self.flat["cutoff"])
            kinds = self.polar[pairs].sum(1)
            swap = (kinds == 1) & self.polar[pairs[:, 1]]
            pairs[swap] = pairs[swap].flip(1)  # the polarisable site first
            self.lists = [pairs[kinds == k] for k in range(3)]
        self.solve(np.ptp(polarity, axis=1).max() > 0)

    def parts(self, kind):
        """One list (by its number of polarisable sites) in parts: (pairs, those of a molecule, separation vectors)."""
        for a in range(0, len(self.lists[kind]), CHUNK):
            pairs = self.lists[kind][a:a + CHUNK]
            d = self.pos[pairs[:, 0]] - self.pos[pairs[:, 1]]
            if self.box is not None:
                d = d - self.box * torch.floor(d.detach() / self.box + 0.5)
            # the 1-2 and 1-3 neighbours of a water are its other two atoms, at scale 0
            own = torch.div(pairs, 3, rounding_mode="floor")
            yield pairs, (own[:, 0] == own[:, 1]).to(torch.float64), d

    def damped(self, pairs, d):
        """The damped dipole interaction tensors [.., 3, 20] of pairs of polarisable sites."""
        r = d.norm(dim=1)
        size = torch.ones(len(self.pos), dtype=torch.float64, device=self.device)
        size = size.index_put((self.sites,), self.leaves[4].reshape(-1, 3)[self.sites].mean(1) ** (1.0 / 6.0))
        screened, bare = _radial(r, self.alpha, 4)
        damp = _thole(self.leaves[6] * r / (size[pairs[:, 0]] * size[pairs[:, 1]]))
        return _tensor(d, [s - (1 - f) * b for s, b, f in zip(screened, bare, damp)])[:, PAIR[1:4]]

    def real_energy(self, kind, pairs, own, d, moments, dipoles, couplings):
        """Real-space energy of some pairs: permanent, permanent with induced, and -u.T.v/2 for each coupling (u, v)."""
        sign = torch.tensor(SIGN, dtype=torch.float64, device=self.device)
        screened, bare = _radial(d.norm(dim=1), self.alpha, (0, 3, 6)[kind])
        g = [s - own * b for s, b in zip(screened, bare)]
        mi, mj = moments[pairs[:, 0]], moments[pairs[:, 1]]
        if kind == 0:
            return COULOMB * (mi[:, 0] * mj[:, 0] * g[0]).sum(), 0.0
        ui, uj = dipoles[pairs[:, 0]], dipoles[pairs[:, 1]]
        if kind == 1:
            mi = torch.cat([mi[:, :1], mi[:, 1:4] + ui, mi[:, 4:]], 1)
            return COULOMB * ((_tensor(d, g) * mi).sum(1) * mj[:, 0]).sum(), 0.0
        energy = torch.einsum("na,nab,nb->", mi, _tensor(d, g)[:, PAIR], mj * sign)
        t = self.damped(pairs, d)
        energy = energy + torch.einsum("ni,nij,nj->", ui, t, mj * sign) - torch.einsum("ni,nij,nj->", uj, t, mi)
        coupled = 0.0
        for u, v in couplings:
            for a, b in ((u, v), (v, u)):
                coupled = coupled - 0.5 * torch.einsum("ni,nij,nj->", a[pairs[:, 0]], t[:, :, 1:4], b[pairs[:, 1]])
        return COULOMB * energy, COULOMB * coupled

    def wide(self, dipoles):
        return torch.nn.functional.pad(dipoles, (1, 16))

    def mesh_energy(self, factor, u, v):
        """factor/2 times the reciprocal-space product of moments u and v, with its derivatives."""
        value, sides = 0.0, ((u, v),) if u is v else ((u, v), (v, u))
        for a, b in sides:
            grid = self.mesh.potential(self.pos.detach(), b.detach())
            for k in range(0, len(self.pos), 32768):
                part = (self.mesh.derivatives(self.pos[k:k + 32768], grid) * a[k:k + 32768]).sum()
                (factor / len(sides) * COULOMB * part).backward(retain_graph=True)
                value += 0.5 * factor / len(sides) * COULOMB * part.item()
        return value

    def permanent_field(self, moments):
        field = torch.zeros_like(self.pos)
        for kind in (1, 2):
            for pairs, own, d in self.parts(kind):
                dipoles = torch.zeros(len(self.pos), 3, dtype=torch.float64, device=self.device, requires_grad=True)
                energy, _ = self.real_energy(kind, pairs, own, d.detach(), moments, dipoles, [])
                field = field - torch.autograd.grad(energy, dipoles)[0] / COULOMB
        return field + self.mesh_field(moments)

    def mesh_field(self, moments):
        """Reciprocal-space and self field of moments (or of dipoles alone)."""
        if self.mesh is None:
            return torch.zeros_like(self.pos)
        with torch.no_grad():
            grid = self.mesh.potential(self.pos, moments)
            field = torch.cat([-self.mesh.derivatives(self.pos[k:k + 32768], grid)[:, 1:4]
                               for k in range(0, len(self.pos), 32768)])
            return field + 4 * self.alpha ** 3 / (3 * SQRT_PI) * moments[:, 1:4]

    def solve(self, anisotropic):
        flat, n, kind = self.flat, len(self.pos), self.flat["polarization"]
        axes = _frames(self.pos, flat)
        moments = _moments(axes, *self.leaves[:4])
        alpha = torch.einsum("nia,ni,nib->nab", axes, self.leaves[4].reshape(n, 3), axes)
        inverse = torch.einsum("nia,ni,nib->nab", axes[self.sites], 1 / self.leaves[4].reshape(n, 3)[self.sites],
                               axes[self.sites])
        fixed = moments.detach().requires_grad_(True)
        e0 = self.permanent_field(fixed.detach())
        polarise = lambda e: torch.einsum("nab,nb->na", alpha.detach(), e)  # noqa: E731
        with torch.no_grad():
            tensors = [(pairs, self.damped(pairs, d)[:, :, 1:4].clone()) for pairs, _, d in self.parts(2)]

            def induced_field(u):
                out = self.mesh_field(self.wide(u))
                for pairs, t in tensors:
                    out.index_add_(0, pairs[:, 0], torch.einsum("nij,nj->ni", t, u[pairs[:, 1]]))
                    out.index_add_(0, pairs[:, 1], torch.einsum("nij,nj->ni", t, u[pairs[:, 0]]))
                return torch.where(self.polar[:, None], out, torch.zeros_like(out))

            mu = polarise(e0)
            couplings, orders = [], [mu]
            if kind == MPIDForce.Mutual:
                def operator(u):
                    out = -induced_field(u)
                    out[self.sites] += torch.einsum("nab,nb->na", inverse, u[self.sites])
                    return out
                r = torch.where(self.polar[:, None], e0, torch.zeros_like(e0)) - operator(mu)
                z = polarise(r)
                p, rz = z.clone(), (r * z).sum()
                stop = 1e-26 * (e0 * mu).sum()
                for _ in range(60):
                    if rz <= stop:
                        break
                    ap = operator(p)
                    step = rz / (p * ap).sum()
                    mu, r = mu + step * p, r - step * ap
                    z = polarise(r)
                    old, rz = rz, (r * z).sum()
                    p = z + rz / old * p
                couplings = [(mu, mu)]
            elif kind == MPIDForce.Extrapolated:
                c = np.cumsum(flat["extrapolation_coefficients"][::-1])[::-1]
                fields = [e0]
                for _ in range(len(c) - 1):
                    fields.append(induced_field(orders[-1]))
                    orders.append(polarise(fields[-1]))
                mu = sum(float(w) * u for w, u in zip(c, orders))
                couplings = [(sum(float(c[k + m + 1]) * orders[k] for k in range(len(c) - 1 - m)), orders[m])
                             for m in range(len(c) - 1)]
            del tensors
        self.dipoles = mu
        # permanent energy and coupling to the dipoles, then the dipoles among themselves
        base, pol = 0.0, 0.5 * COULOMB * (mu * e0).sum().item()
        for k in range(3):
            for pairs, own, d in self.parts(k):
                energy, coupled = self.real_energy(k, pairs, own, d, fixed, mu, couplings)
                (energy + coupled).backward(retain_graph=True)
                base += energy.item()
        if self.mesh is not None:
            total = fixed + self.wide(mu)
            base += self.mesh_energy(1.0, total, total)
            w = self.wide(mu)
            base += self.mesh_energy(-1.0, w, w)
            for u, v in couplings:
                self.mesh_energy(1.0, w if u is mu else self.wide(u), w if v is mu else self.wide(v))
            order = torch.tensor([sum(p) for p in POWERS[:20]], device=self.device)
            scale = torch.tensor([1.0, 2 / 3, 4 / 15 * 6, 8 / 105 * 90], dtype=torch.float64, device=self.device)
            power = self.alpha ** (2.0 * order)
            squares = (fixed ** 2 / torch.tensor(WEIGHT, dtype=torch.float64, device=self.device) * power *
                       scale[order]).sum() + 4 / 3 * self.alpha ** 2 * (fixed[:, 1:4] * mu).sum()
            own = -self.alpha * COULOMB / SQRT_PI * squares
            own.backward()
            base += own.item()
        self.energy = base + pol
        # the polarisability: its molecular axes turn with the atoms
        if kind == MPIDForce.Extrapolated:
            top = len(orders)
            elastic = sum(-0.5 * float(c[k + m]) * torch.einsum("na,nab,nb->", fields[k], alpha, fields[m])
                          for k in range(top) for m in range(top - k))
        else:
            elastic = 0.5 * torch.einsum("na,nab,nb->", mu[self.sites], inverse, mu[self.sites])
        rest = COULOMB * elastic + (moments * fixed.grad).sum()
        if kind == MPIDForce.Mutual and anisotropic:
            rest = rest - self.convention(axes, mu)
        rest.backward()
        self.forces = -self.pos.grad

    def convention(self, axes, mu):
        """The evaluator follows the reference in leaving out half of the torque about the pair axis between two
        induced dipoles (unless asked for conservative torques): the work of what is left out, for turning frames."""
        torque = torch.zeros_like(self.pos)
        with torch.no_grad():
            for pairs, _, d in self.parts(2):
                f = -self.damped(pairs, d)[:, :, 1:4]
                z = -d / d.norm(dim=1, keepdim=True)
                x = torch.zeros_like(z)
                x[:, 0] = 1.0
                x = x - z * z[:, :1]
                x = x / x.norm(dim=1, keepdim=True)
                y = torch.linalg.cross(z, x)
                f = torch.einsum("ni,nij,nj->n", x, f, x)
                ui, uj = mu[pairs[:, 0]], mu[pairs[:, 1]]
                for k, (a, b) in enumerate(((ui, uj), (uj, ui))):
                    torque.index_add_(0, pairs[:, k], -COULOMB * z * (f * (a * y).sum(1) * (b * x).sum(1))[:, None])
        turned = 0.5 * torch.linalg.cross(axes.detach(), axes).sum(1)
        return (torque * turned).sum()


def exact(case, seed):
    if case["kind"] == "batch":
        found = [_Exact(*system) for system in _batch_systems(case, seed)]
        return dict(energies=np.array([e.energy for e in found]), forces=torch.cat([e.forces for e in found]))
    force, pos, box = _system(case, seed)
    found = _Exact(force, pos, box)
    if case["kind"] == "gradients":
        grads = [torch.zeros_like(t) if t.grad is None else t.grad for t in found.leaves]
        grads[1].reshape(len(pos), -1)[~found.polar] = 0.0  # bare charges have no other gradients
        shaped = [_rows(g, len(pos)) for g in grads[:-1]] + grads[-1:]
        out = dict(energy=found.energy, **dict(zip(PARAMETERS + ("default_thole",), shaped)))
        # the energy is defined for traceless tensors only: their components' gradients have a free trace part
        return dict(out, quadrupoles=None, octopoles=None)
    out = dict(energy=found.energy, forces=found.forces)
    if case["dipoles"]:
        out["dipoles"] = found.dipoles
    return out
