"""Timed cases: what a program built on inq_amd has the library do.

Every case goes through the public entry points on device-resident states, as
the ground-state and real-time loops call them: H on one block, on a batch of
k-points and in the reference's point-major layout, real-time steps, the
steepest-descent eigensolver, a hybrid functional's H, orthogonalisation, the
ACE build, exchange between k-points and the density / Hartree update.

Systems: orthorhombic cells with Gaussian local potentials and Gaussian
Kleinman-Bylander projectors on every atom.  The listed sizes are the
benchmark configurations (8-atom diamond cell on 32^3, 64-atom Si on 72^3,
4-atom fcc Al on 24^3 with 64 k-points, the 432-state block of 216-atom Si at
its sphere size) and one slab with three different axes; draw() spreads grids,
state counts, precisions, k-points, projector channels and layouts over the
ranges in between.

States are random with coefficients that decay with the kinetic energy, as
those of converged or partly converged orbitals do.  exact() computes the same
results in complex128 with torch's FFTs and numpy's dense algebra alone.
"""
import ctypes
import math

import numpy as np
import torch

from inq_amd import Context, DeviceArray, KSHamiltonian
from inq_amd import eigensolvers, operations
from inq_amd.exchange import ExchangeOperator
from inq_amd.real_time import Propagator

# line lengths the library builds, up to the largest benchmark grid
SIZES = (16, 18, 20, 24, 28, 30, 32, 36, 40, 48, 54, 60, 64, 72, 80, 96)
C64, C128 = "complex64", "complex128"
TDT = {C64: torch.complex64, C128: torch.complex128}
NDT = {C64: np.complex64, C128: np.complex128}
POINT_MAJOR = KSHamiltonian.SPHERE_POINT
V_DEPTH = -4.0  # Hartree, depth of the Gaussian local potential of an atom
DT = 0.05       # real-time step, atomic time units
KICK = -0.01    # velocity-gauge kick along x


# ------------------------------------------------------------------ cases

def _case(name, kind, n, cell, ecut, nst, dtype, **more):
    c = {"kind": kind, "n0": n[0], "n1": n[1], "n2": n[2], "a0": cell[0], "a1": cell[1], "a2": cell[2],
         "ecut": ecut, "nst": nst, "dtype": dtype, "atoms": 0, "sites": "random", "nlm": 4, "width": 0.9,
         "sigma": 0.7, "k0": 0.0, "k1": 0.0, "k2": 0.0}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    si64 = {"n": (72, 72, 72), "cell": (20.52, 20.52, 20.52), "ecut": 30.0, "nst": 128}
    si = {"sites": "diamond", "atoms": 64}
    return [
        # the smallest block: the 8-atom cell, where launches and latency count
        _case("h_c8_fp64", "h", (32, 32, 32), (6.74, 6.74, 6.74), 25.0, 16, C128, sites="diamond", atoms=8,
              sigma=0.6, width=0.8),
        # every (k-point, spin) block of a small metal in one call, spheres of uneven size
        _case("h_kpoints_batch", "batch", (24, 24, 24), (7.65, 7.65, 7.65), 20.0, 12, C64, sites="fcc", atoms=4, nk=4),
        # the headline: H on the 128 states of 64-atom Si, mixed precision and double
        _case("h_si64_fp32", "h", dtype=C64, **si64, **si),
        _case("h_si64_fp64", "h", dtype=C128, **si64, **si),
        # a slab: three different axes, an odd state count, a k-point, s + p + d projectors,
        # states in the reference's point-major layout
        _case("h_slab_layout", "h", (40, 48, 60), (11.2, 13.6, 17.1), 28.0, 37, C64, atoms=22, nlm=9, layout=1,
              k0=0.7, k1=-1.1, k2=0.3),
        # real-time propagation after a kick, the step captured in a graph, records read after two steps
        _case("etrs_si64", "etrs", dtype=C64, steps=2, **si64, **si),
        # one eigensolver call of the ground-state loop: five line minimisations, orthogonalisation
        _case("descent_si64", "descent", dtype=C64, **si64, **si),
        # H of a hybrid functional: H, then the ACE projectors' exchange, in double
        _case("hybrid_si64", "hybrid", dtype=C128, **si64, **si),
        # orthogonalisation of a large block: 432 states on the sphere of 216-atom Si
        _case("orthogonalize_432", "orth", (96, 96, 96), (30.78, 30.78, 30.78), 30.0, 432, C64),
        # hybrid functional: every pair density of the block, then the ACE projectors
        _case("ace_si64", "ace", dtype=C64, **si64, **si),
        # exchange of one k-point's states with those of eight k-points, in double
        _case("exchange_kpoints", "xk", (24, 24, 24), (7.65, 7.65, 7.65), 20.0, 12, C128, nk=8),
        # the density of a block and its Hartree potential and energy: the update of a self-consistent step
        _case("density_hartree", "scf", dtype=C128, **{**si64, "nst": 96}),
    ]


def _size(rng, lo, hi):
    """a built line length between lo and hi, spread over the logarithm"""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min((s for s in SIZES if lo <= s <= hi), key=lambda s: abs(s - x))


def _grid(rng, lo, hi):
    """half cubes, half cells whose axes differ by up to half"""
    n = _size(rng, lo, hi)
    if rng.random() < 0.5:
        return (n, n, n)
    return tuple(_size(rng, max(lo, int(n / 1.3)), min(hi, int(n * 1.3) + 1)) for _ in range(3))


def _count(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["h", "h", "h", "batch", "etrs", "descent", "hybrid", "orth", "ace", "xk", "scf"])
    top = {"batch": 32, "xk": 32, "ace": 64}.get(kind, 80)
    n = _grid(rng, 16 if kind in ("h", "xk", "batch") else 24, top)
    points = n[0] * n[1] * n[2]
    spacing = rng.uniform(0.24, 0.31)
    cell = tuple(round(x * spacing * rng.uniform(0.98, 1.02), 4) for x in n)
    ecut = round(0.5 * (rng.uniform(0.62, 0.72) * math.pi / spacing) ** 2, 3)
    # at most the largest listed block's points times states
    most = int(72 ** 3 * 128 / points)
    nst = {"h": (3, 160), "batch": (4, 16), "etrs": (8, 96), "descent": (8, 160), "hybrid": (8, 144),
           "orth": (24, 320), "ace": (6, 64), "xk": (4, 20), "scf": (4, 128)}[kind]
    nst = _count(rng, nst[0], max(nst[0], min(nst[1], most)))
    dtype = rng.choice([C64, C128])
    if kind in ("xk", "scf"):  # small grids, and the FP64 density, run in double
        dtype = C128
    if kind == "ace":
        dtype = C64
    more = {"atoms": max(1, round(cell[0] * cell[1] * cell[2] / rng.uniform(100.0, 140.0)))}
    if kind in ("batch", "xk"):
        more["nk"] = rng.choice([2, 3]) if kind == "batch" else rng.choice([2, 3, 5, 8])
    if kind == "etrs":
        more["steps"] = rng.choice([1, 2])
    if kind == "h":
        more["layout"] = rng.choice([0, 0, 0, 1])
        more["nlm"] = rng.choice([1, 4, 4, 9] if dtype == C64 else [1, 4])
    if kind in ("h", "descent", "hybrid", "etrs", "scf") and rng.random() < 0.5:
        more.update({k: round(rng.uniform(-1.5, 1.5), 3) for k in ("k0", "k1", "k2")})
    return _case(None, kind, n, cell, ecut, nst, dtype, **more)


# ------------------------------------------------------------------ the system of a case

def _n(case):
    return case["n0"], case["n1"], case["n2"]


def _cell(case):
    return case["a0"], case["a1"], case["a2"]


def _volume(case):
    return case["a0"] * case["a1"] * case["a2"]


def _points(case):
    return case["n0"] * case["n1"] * case["n2"]


def _vol_el(case):
    """volume element of the G sphere, V / N^2"""
    return _volume(case) / float(_points(case)) ** 2


def _positions(case, seed):
    """[atoms, 3] bohr: diamond or fcc conventional cells, or random sites (off the grid points, where
    the direction from an atom to its own grid point would be rounding)"""
    cell = np.array(_cell(case))
    if case["sites"] == "random":
        rng, pos = np.random.default_rng(seed + 17), np.zeros((0, 3))
        for _ in range(case["atoms"]):  # the farthest of 20 places from the atoms so far, as atoms keep apart
            x = rng.uniform(-0.5, 0.5, (20, 1, 3))
            d = x - pos
            far = np.min(np.sum(((d - np.round(d)) * cell) ** 2, axis=2), axis=1, initial=1e9)
            pos = np.concatenate([pos, x[np.argmax(far)]])
        return pos * cell
    sites = [(0, 0, 0), (0, .5, .5), (.5, 0, .5), (.5, .5, 0)]
    if case["sites"] == "diamond":
        sites += [(.25, .25, .25), (.25, .75, .75), (.75, .25, .75), (.75, .75, .25)]
    rep = round((case["atoms"] / len(sites)) ** (1.0 / 3.0))
    cells = [(i, j, k) for i in range(rep) for j in range(rep) for k in range(rep)]
    return np.array([(np.array(s) + c) / rep for c in cells for s in sites]) * cell + (0.031, 0.017, 0.043)


def _couplings(case, seed):
    rng = np.random.default_rng(seed + 1000)
    return [np.diag(rng.uniform(-2.0, 2.0, case["nlm"])) for _ in range(case["atoms"])]


def _axis(n, a):
    """positions along one axis in the symmetric range, as the grid stores them"""
    i = np.arange(n)
    return np.where(i >= (n + 1) // 2, i - n, i) / n * a


def _potential(case, seed):
    """sum of the atoms' Gaussians at the nearest image, host [N] float64"""
    pos = _positions(case, seed)
    g = []
    for d, (n, a) in enumerate(zip(_n(case), _cell(case))):
        x = _axis(n, a)[None, :] - pos[:, d:d + 1]
        x -= np.round(x / a) * a
        g.append(np.exp(-x * x / (2.0 * case["sigma"] ** 2)))
    plane = (g[0][:, :, None] * g[1][:, None, :]).reshape(len(pos), case["n0"] * case["n1"])
    return V_DEPTH * (plane.T @ g[2]).reshape(-1)


def _sphere(case, k, ecut):
    """flattened FFT indices with |G + k|^2 / 2 < ecut, ascending, and |G + k|^2 / 2 there"""
    g2 = []
    for n, a, kd in zip(_n(case), _cell(case), k):
        i = torch.arange(n, dtype=torch.float64, device="cuda")
        m = torch.where(i >= (n + 1) // 2, i - n, i)
        g2.append(((2.0 * math.pi * m + kd) / a) ** 2)
    kin = 0.5 * (g2[0][:, None, None] + g2[1][None, :, None] + g2[2][None, None, :]).reshape(-1)
    idx = torch.nonzero(kin < ecut).reshape(-1)
    return idx, kin[idx]


def _raw_states(kin, nst, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    c = torch.view_as_complex(torch.randn((nst, kin.numel(), 2), dtype=torch.float64, device="cuda", generator=gen))
    return c * (1.0 + 0.5 * kin) ** -1.5


def _orthonormal(c, vol_el):
    """c <- conj(L)^-1 c with the overlap S = vol_el conj(c) c^T = L L^H, on the host"""
    c = c.cpu().numpy()
    return _solve_rows(vol_el * (c.conj() @ c.T), c)


def _solve_rows(m, c):
    """conj(L)^-1 c with m = L L^H, numpy"""
    L = np.linalg.cholesky(0.5 * (m + m.conj().T))
    return torch.from_numpy(np.linalg.inv(L).conj() @ c)


def _states(case, kin, seed):
    """normalised states; random ones of this many coefficients are nearly orthogonal"""
    c = _raw_states(kin, case["nst"], seed)
    norm = torch.sqrt(_vol_el(case) * torch.sum(c.real ** 2 + c.imag ** 2, dim=1, keepdim=True))
    return (c / norm).to(TDT[case["dtype"]])


def _projectors(case, c):
    """ACE projectors of the size exchange gives them: the states, shifted by one and smoothed"""
    return 0.3 * torch.roll(c, 1, dims=0) + 0.2 * torch.roll(c, 2, dims=0)


def _kvec(case):
    return case["k0"], case["k1"], case["k2"]


def _blocks(case):
    """(k, spin, ecut) of every block of a batch: an nk^3 Monkhorst-Pack grid x 2 spins, cutoffs 5% apart"""
    nk = case["nk"]
    jit = np.random.default_rng(2003).uniform(-0.05, 0.05, 2 * nk ** 3)
    out = []
    for i in range(nk ** 3):
        f = [(j if 2 * j < nk else j - nk) / nk for j in (i // (nk * nk), i // nk % nk, i % nk)]
        for s in range(2):
            out.append((tuple(2.0 * math.pi * x for x in f), s, case["ecut"] * (1.0 + jit[2 * i + s])))
    return out


def _hf_points(case):
    """the k-points of an exchange case: nk points along the cell's diagonal, the first being phi's"""
    return [tuple(2.0 * math.pi * x * j / case["nk"] for x in (0.5, 0.3, -0.4)) for j in range(case["nk"])]


def _zeroterm(case):
    """the Poisson value at G = 0 of a spherical cutoff of the cell's volume: 2 pi R^2"""
    return 2.0 * math.pi * (3.0 * _volume(case) / (4.0 * math.pi)) ** (2.0 / 3.0)



class _Shared(DeviceArray):
    """a torch tensor's memory as a device array: the library takes the caller's pointers"""

    def __init__(self, ctx, tensor):
        self.ctx = ctx
        self.tensor = tensor
        self.shape = tuple(tensor.shape)
        self.dtype = np.dtype(str(tensor.dtype).split(".")[1])
        self.nbytes = tensor.numel() * tensor.element_size()
        self.ptr = ctypes.c_void_p(tensor.data_ptr())

    def free(self):
        pass


def _hamiltonian(ctx, case, seed, spins=1):
    h = KSHamiltonian(ctx, np.diag(_cell(case)), _n(case))
    v = _potential(case, seed)
    if spins == 2:
        h.set_scalar_potential(np.stack([v, 0.9 * v + 0.1], axis=1), ncomp=2)
    else:
        h.set_scalar_potential(v)
    for p, d in zip(_positions(case, seed), _couplings(case, seed)):
        h.add_projector(p, 2.0, case["nlm"], d, width=case["width"])
    return h


def _basis(h, k, ecut, states, spin=0):
    b = h.basis(k, ecut, spin)
    if b.npw != states.shape[1]:
        raise ValueError("the G sphere of the case lies on a rounding boundary")
    return b


# ------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    """the Hamiltonian, bases, states and output arrays that a program holds"""
    ctx = Context(0)
    kind, nst, dt = case["kind"], case["nst"], TDT[case["dtype"]]
    s = {"case": case, "ctx": ctx}
    if kind == "orth":
        idx, kin = _sphere(case, _kvec(case), case["ecut"])
        s["phi"] = _Shared(ctx, _raw_states(kin, nst, seed).to(dt))
        return s
    s["ham"] = h = _hamiltonian(ctx, case, seed, 2 if kind == "batch" else 1)
    if kind == "batch":
        s["bases"], s["psi"], s["out"] = [], [], []
        for i, (k, spin, ecut) in enumerate(_blocks(case)):
            c = _states(case, _sphere(case, k, ecut)[1], seed + 31 * i)
            s["bases"].append(_basis(h, k, ecut, c, spin))
            s["psi"].append(_Shared(ctx, c))
            h.prepare(s["bases"][-1], nst, NDT[case["dtype"]])
        # the blocks' results one after another in one array
        s["flat"] = torch.empty(sum(c.tensor.numel() for c in s["psi"]), dtype=dt, device="cuda")
        for c, out in zip(s["psi"], s["flat"].split([c.tensor.numel() for c in s["psi"]])):
            s["out"].append(_Shared(ctx, out.view(c.shape)))
        return s
    if kind == "xk":
        s["hf"] = []
        for j, q in enumerate(_hf_points(case)):
            c = _states(case, _sphere(case, q, case["ecut"])[1], seed + 31 * j)
            b = _basis(h, q, case["ecut"], c)
            s["hf"].append((b, _Shared(ctx, c), np.linspace(2.0, 1.0, nst), _zeroterm(case) if j == 0 else 0.0))
        s["basis"], s["phi"] = s["hf"][0][:2]
        s["out"] = _Shared(ctx, torch.empty_like(s["phi"].tensor))
        s["exx"] = ExchangeOperator(h, s["basis"], 0.25)
        return s
    k = _kvec(case)
    c = _states(case, _sphere(case, k, case["ecut"])[1], seed)
    s["basis"] = b = _basis(h, k, case["ecut"], c)
    if kind == "etrs":
        h.uniform_vector_potential = np.array([KICK * case["a0"], 0.0, 0.0])
    point = bool(case.get("layout", 0))
    s["phi"] = _Shared(ctx, c.t().contiguous() if point else c)
    h.prepare(b, nst, NDT[case["dtype"]])
    if kind == "h":
        s["out"] = _Shared(ctx, torch.empty_like(s["phi"].tensor))
    elif kind == "etrs":
        s["prop"] = Propagator(h, [b], [s["phi"]], [np.full(nst, 2.0)], DT, ring_capacity=64)
    elif kind == "hybrid":
        s["out"] = _Shared(ctx, torch.empty_like(c))
        s["exx"] = ExchangeOperator(h, b, 0.25, 0.0)
        s["exx"].xi = _Shared(ctx, _projectors(case, c))
    elif kind == "ace":
        s["exx"] = ExchangeOperator(h, b, 0.25, _zeroterm(case))
        s["exx"].xi = _Shared(ctx, torch.empty_like(c))
        s["occ"] = np.full(nst, 2.0)
    elif kind == "scf":
        n = _points(case)
        s["occ"] = np.full(nst, 2.0)
        s["rho"] = _Shared(ctx, torch.zeros(n, dtype=torch.float64, device="cuda"))
        s["vh"] = _Shared(ctx, torch.zeros(n, dtype=torch.float64, device="cuda"))
    return s


def run(s):
    """one pass, as a program calls it"""
    case = s["case"]
    kind = case["kind"]
    if kind == "h":
        if case.get("layout", 0):
            s["ham"].apply_layout(s["basis"], s["phi"], s["out"], POINT_MAJOR)
        else:
            s["ham"].apply(s["basis"], s["phi"], s["out"])
        return s["out"].tensor
    if kind == "batch":
        s["ham"].apply_batch(s["bases"], s["psi"], s["out"])
        return s["flat"]
    if kind == "etrs":
        s["prop"].step(case["steps"], graph=True)
        # the records are float64 sums over states of the case's precision
        rec = s["prop"].records(cap=case["steps"])
        return {"phi": s["phi"].tensor, "records": rec.astype(np.float32) if case["dtype"] == C64 else rec}
    if kind == "descent":
        eigensolvers.steepest_descent(s["ham"], s["basis"], s["phi"])
        return s["phi"].tensor
    if kind == "hybrid":
        s["ham"].apply(s["basis"], s["phi"], s["out"])
        s["exx"].ace(s["phi"], s["out"])
        return s["out"].tensor
    if kind == "orth":
        operations.orthogonalize(s["ctx"], s["phi"], _vol_el(case))
        return s["phi"].tensor
    if kind == "ace":
        e = s["exx"].update(s["phi"], s["occ"])
        return {"energy": np.float32(e), "xi": s["exx"].xi.tensor}
    if kind == "xk":
        s["out"].tensor.zero_()
        s["exx"].direct_kpts(s["phi"], s["hf"], exxphi=s["out"])
        return s["out"].tensor
    s["rho"].tensor.zero_()
    s["ham"].density_add(s["basis"], s["phi"], s["occ"], density=s["rho"])
    vh, e = s["ham"].hartree(s["rho"], s["vh"])
    return {"density": s["rho"].tensor, "vh": vh.tensor, "energy": e}


# ------------------------------------------------------------------ work

def _h_flops(case, npw, natoms):
    """one H on one state: two transforms pruned to the sphere, potential, projectors, kinetic"""
    n0, n1, n2 = _n(case)
    f = min(1.0, (6.0 * npw / (math.pi * _points(case))) ** (1.0 / 3.0))  # sphere diameter over the grid
    fft = sum(lines * 5.0 * n * math.log2(n) for lines, n in
              ((0.785 * f * f * n0 * n1, n2), (f * n0 * n2, n1), (n1 * n2, n0)))
    sphere = 4.0 / 3.0 * math.pi * 8.0 / _volume(case) * _points(case)  # points of a projector sphere, r = 2
    return 2.0 * fft + 2.0 * _points(case) + natoms * sphere * case["nlm"] * 8.0 + 4.0 * npw


def _npw(case, ecut=None):
    """points of the G sphere, from its volume"""
    return _volume(case) * (2.0 * (ecut or case["ecut"])) ** 1.5 / (6.0 * math.pi ** 2)


def work(case):
    kind, nst = case["kind"], case["nst"]
    s = 8 if case["dtype"] == C64 else 16
    npw, n = _npw(case), _points(case)
    state = nst * npw * s
    tables = n * s / 2 + npw * s / 2
    h = nst * _h_flops(case, npw, case["atoms"])
    pair = 2.0 * 5.0 * n * math.log2(n) + 16.0 * n  # one Poisson solve and its products
    mm = 8.0 * nst * nst * npw                      # one dense product of the block with an nst x nst matrix
    if kind == "h":
        return {"bytes": 2 * state + tables, "flops": h}
    if kind == "batch":
        blocks = 2 * case["nk"] ** 3
        return {"bytes": blocks * (2 * state + npw * s / 2) + n * s, "flops": blocks * h}
    if kind == "etrs":
        return {"bytes": 2 * state + tables, "flops": case["steps"] * (9 * h + 8 * 8.0 * nst * npw)}
    if kind == "descent":
        return {"bytes": 2 * state + tables, "flops": 6 * h + 5 * 80.0 * nst * npw + mm + 8.0 * nst ** 3}
    if kind == "hybrid":
        return {"bytes": 3 * state + tables, "flops": h + 2 * mm}
    if kind == "orth":
        # the overlap is Hermitian and the rotation triangular: half of each product
        return {"bytes": 2 * state, "flops": mm + 8.0 * 2.0 / 3.0 * nst ** 3}
    if kind == "ace":
        return {"bytes": 2 * state, "flops": nst * (nst + 1) / 2 * pair + 1.5 * mm}
    if kind == "xk":
        return {"bytes": (case["nk"] + 2) * state, "flops": case["nk"] * nst * nst * pair}
    return {"bytes": state + 3 * 8.0 * n, "flops": nst * 5.0 * n * math.log2(n) + 10.0 * n * math.log2(n)}


# ------------------------------------------------------------------ results in 64 bits

def _harmonic(l, x, y, z, r2):
    """real spherical harmonics: s; p in the order y, z, x; d in the order xy, yz, 3z^2 - r^2, xz, x^2 - y^2"""
    if l == 0:
        return np.full_like(x, 0.5 / math.sqrt(math.pi))
    safe = np.where(r2 > 0.0, r2, 1.0)
    if l <= 3:
        v = math.sqrt(3.0 / (4.0 * math.pi)) * (y, z, x)[l - 1] / np.sqrt(safe)
    else:
        d = (x * y, y * z, (3.0 * z * z - r2) / (2.0 * math.sqrt(3.0)), x * z, 0.5 * (x * x - y * y))[l - 4]
        v = math.sqrt(15.0 / (4.0 * math.pi)) * d / safe
    return np.where(r2 > 0.0, v, 0.0)


def _transform(f, u, n):
    """3-D transforms of rows [m, N], 32 at a time"""
    return torch.cat([f(x.reshape(-1, *n), dim=(1, 2, 3)).reshape(x.shape) for x in u.split(32)])


class _Exact:
    """H = kinetic + local + Kleinman-Bylander on complex128 sphere coefficients [nst, npw]"""

    def __init__(self, case, seed, k, ecut, kick=0.0, shared=None):
        self.case = case
        self.n, self.vol = _n(case), _volume(case)
        kk = (k[0] + kick * case["a0"], k[1], k[2])
        self.idx, _ = _sphere(case, k, ecut)
        self.kin = self._kinetic(kk)
        self.v = shared.v if shared else torch.from_numpy(_potential(case, seed)).cuda()
        self.points = shared.points if shared else self._projectors(seed)
        self.phase = [torch.exp(1j * sum(r[:, d] * kk[d] for d in range(3))) for _, _, r, _ in self.points]

    def _kinetic(self, kk):
        f = self.idx
        n0, n1, n2 = self.n
        kin = torch.zeros(f.numel(), dtype=torch.float64, device="cuda")
        for i, n, a, kd in zip((f // (n1 * n2), f // n2 % n1, f % n2), self.n, _cell(self.case), kk):
            m = torch.where(i >= (n + 1) // 2, i - n, i).double()
            kin += 0.5 * ((2.0 * math.pi * m + kd) / a) ** 2
        return kin

    def _projectors(self, seed):
        """per atom: grid indices, values [nlm, points], float32-rounded fractional positions, couplings"""
        case, out = self.case, []
        cell = np.array(_cell(case))
        grids = [_axis(n, a) for n, a in zip(self.n, cell)]
        for p, d in zip(_positions(case, seed), _couplings(case, seed)):
            near = []
            for x, a, pd in zip(grids, cell, p):
                dx = x - pd
                dx -= np.round(dx / a) * a
                near.append((np.nonzero(np.abs(dx) <= 2.0)[0], dx))
            i, j, l = (m.reshape(-1) for m in np.meshgrid(*(w for w, _ in near), indexing="ij"))
            r = np.stack([near[0][1][i], near[1][1][j], near[2][1][l]], axis=1)
            keep = np.sum(r * r, axis=1) <= 4.0
            i, j, l, r = i[keep], j[keep], l[keep], r[keep]
            dist = np.sqrt(np.sum(r * r, axis=1)).astype(np.float32).astype(np.float64)
            frac = (r / cell).astype(np.float32).astype(np.float64)
            x, y, z = (frac * cell).T
            radial = np.exp(-dist * dist / (2.0 * case["width"] ** 2))
            b = np.stack([radial * _harmonic(m, x, y, z, x * x + y * y + z * z) for m in range(case["nlm"])])
            at = (i * self.n[1] + j) * self.n[2] + l
            out.append(tuple(torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (at, b, frac, d)))
        return out

    def to_real(self, c):
        u = torch.zeros((c.shape[0], self.v.numel()), dtype=torch.complex128, device="cuda")
        u[:, self.idx] = c
        return _transform(torch.fft.ifftn, u, self.n)

    def to_sphere(self, u):
        return _transform(torch.fft.fftn, u, self.n)[:, self.idx]

    def project(self, u):
        """per atom P = dV sum beta exp(ik.r) u and D P (D is diagonal), [nst, nlm] both"""
        dv = self.vol / self.v.numel()
        out = []
        for (at, b, _, d), ph in zip(self.points, self.phase):
            x = u[:, at] * ph
            p = dv * torch.stack([torch.sum(x * row, dim=1) for row in b], dim=1)
            out.append((p, p * torch.diagonal(d)))
        return out

    def apply(self, c):
        u = self.to_real(c)
        w = u * self.v
        for (at, b, _, _), ph, (_, dp) in zip(self.points, self.phase, self.project(u)):
            w[:, at] += sum(dp[:, m, None] * b[m] for m in range(b.shape[0])) * torch.conj_physical(ph)
        return self.to_sphere(w) + self.kin * c


def _exact_record(e, c, occ, step):
    """the observables of the states: kinetic, eigenvalue sum, non-local, norms, dipole, step"""
    case, n = e.case, e.v.numel()
    norm = torch.sum(c.abs() ** 2, dim=1)
    u = e.to_real(c)
    eig = torch.sum((c.conj() * e.apply(c)).real, dim=1)
    nl = sum(torch.sum((p.conj() * dp).real, dim=1) for p, dp in e.project(u))
    rho = torch.sum(u.abs() ** 2, dim=0).reshape(e.n) * occ
    dip = []
    for d in range(3):
        x = torch.from_numpy(_axis(e.n[d], _cell(case)[d])).cuda()
        dip.append(float(torch.sum(rho * x.reshape([-1 if i == d else 1 for i in range(3)]))) * e.vol / n)
    return [float(torch.sum(occ * torch.sum(e.kin * c.abs() ** 2, dim=1) / norm)), float(torch.sum(occ * eig / norm)),
            float(torch.sum(occ * nl)), float(torch.sum(norm)) * _vol_el(case), *dip, float(step)]


def _exact_descent(case, e, c):
    vol = _vol_el(case)
    dot = lambda a, b: vol * torch.sum(a.conj() * b, dim=1, keepdim=True)  # noqa: E731
    g2h = _Exact._kinetic(e, (0.0, 0.0, 0.0))
    hc = e.apply(c)
    for _ in range(5):
        m4, m5 = dot(hc, c), dot(c, c)
        r = hc - m4 / m5.real * c
        t = (torch.sum(g2h * r.abs() ** 2, dim=1) / torch.sum(r.abs() ** 2, dim=1))[:, None]
        x = g2h / t
        top = ((8.0 * x + 12.0) * x + 18.0) * x + 27.0
        r = r * (top / (top + 16.0 * x ** 4))
        hr = e.apply(r)
        m0, m1, m2, m3 = dot(r, r), dot(c, r), dot(r, hr), dot(c, hr)
        ca, cb, cc = (m0 * m3 - m2 * m1).real, (m5 * m2 - m4 * m0).real, (m4 * m1 - m3 * m5).real
        den = cb + torch.sqrt(cb * cb - 4.0 * ca * cc)
        lam = torch.where(den.abs() < 1e-15, torch.zeros_like(den), 2.0 * cc / den)
        c, hc = c + lam * r, hc + lam * hr
    return _orthonormal(c, vol)


def _poisson(case, rho, shift, zeroterm):
    """potential of densities [m, N]: 4 pi / |G + q|^2, zeroterm at G + q = 0"""
    g2 = []
    for n, a, q in zip(_n(case), _cell(case), shift):
        i = torch.arange(n, dtype=torch.float64, device="cuda")
        g2.append(((2.0 * math.pi * torch.where(i >= (n + 1) // 2, i - n, i) + q) / a) ** 2)
    g2 = g2[0][:, None, None] + g2[1][None, :, None] + g2[2][None, None, :]
    kern = torch.where(g2 < 1e-6, torch.full_like(g2, zeroterm), 4.0 * math.pi / g2)
    f = _transform(torch.fft.fftn, rho, _n(case)) * kern.reshape(-1)
    return _transform(torch.fft.ifftn, f, _n(case))


def _exchange(case, e, c, blocks, coeff):
    """sum over blocks (k shift, states, occupations, zeroterm) of coeff occ_j hf_j v[conj(hf_j) phi_i]"""
    u = e.to_real(c)
    w = torch.zeros_like(u)
    for shift, hf, occ, zt in blocks:
        for j in range(hf.shape[0]):
            w += coeff * float(occ[j]) * hf[j] * _poisson(case, hf[j].conj() * u, shift, zt)
    return e.to_sphere(w)


def exact(case, seed):
    kind, nst = case["kind"], case["nst"]
    wide = lambda t: t.to(torch.complex128)  # noqa: E731
    if kind == "orth":
        _, kin = _sphere(case, _kvec(case), case["ecut"])
        c = wide(_raw_states(kin, nst, seed).to(TDT[case["dtype"]]))
        return _orthonormal(c, _vol_el(case))
    if kind == "batch":
        outs, v = [], None
        for i, (k, spin, ecut) in enumerate(_blocks(case)):
            e = _Exact(case, seed, k, ecut, shared=v)
            v = v or e
            base = v.v
            e.v = base if spin == 0 else 0.9 * base + 0.1
            outs.append(e.apply(wide(_states(case, _sphere(case, k, ecut)[1], seed + 31 * i))))
            e.v = base
        return torch.cat([o.reshape(-1) for o in outs])
    if kind == "xk":
        qs = _hf_points(case)
        occ = np.linspace(2.0, 1.0, nst)
        es = [_Exact({**case, "atoms": 0, "sites": "random"}, seed, q, case["ecut"]) for q in qs]
        cs = [wide(_states(case, _sphere(case, q, case["ecut"])[1], seed + 31 * j)) for j, q in enumerate(qs)]
        zero = [_zeroterm(case)] + [0.0] * (len(qs) - 1)
        blocks = [(q, e.to_real(c), occ, z) for q, e, c, z in zip(qs, es, cs, zero)]
        return _exchange(case, es[0], cs[0], blocks, -0.5 * 0.25)
    k = _kvec(case)
    bare = kind in ("ace", "scf")  # no Hamiltonian acts
    e = _Exact({**case, "atoms": 0, "sites": "random"} if bare else case, seed, k, case["ecut"], KICK if kind == "etrs" else 0.0)
    c = wide(_states(case, _sphere(case, k, case["ecut"])[1], seed))
    if kind == "h":
        h = e.apply(c)
        return h.t().contiguous() if case.get("layout", 0) else h
    if kind == "etrs":
        rec = []
        for step in range(case["steps"]):
            for _ in range(2):
                term, out = c, c
                for it in range(1, 5):
                    term = (-0.5j * DT / it) * e.apply(term)
                    out = out + term
                c = out
            rec.append(_exact_record(e, c, 2.0, step))
        return {"phi": c, "records": np.array(rec)}
    if kind == "descent":
        return _exact_descent(case, e, c)
    if kind == "hybrid":
        xi = wide(_projectors(case, c.to(TDT[case["dtype"]]))).cpu().numpy()
        ov = _vol_el(case) * (xi.conj() @ c.cpu().numpy().T)
        return e.apply(c) - torch.from_numpy(np.ascontiguousarray(ov.T) @ xi).cuda()
    if kind == "ace":
        u = e.to_real(c)
        w = _exchange(case, e, c, [((0.0, 0.0, 0.0), u, np.full(nst, 2.0), _zeroterm(case))], 0.5 * 0.25)
        w = w.cpu().numpy()
        m = _vol_el(case) * (w.conj() @ c.cpu().numpy().T)
        return {"energy": -0.5 * 2.0 * float(np.trace(m).real), "xi": _solve_rows(m, w)}
    rho = 2.0 * torch.sum(e.to_real(c).abs() ** 2, dim=0)
    vh = _poisson(case, rho[None].to(torch.complex128), (0.0, 0.0, 0.0), 0.0)[0].real
    return {"density": rho, "vh": vh, "energy": 0.5 * float(torch.sum(rho * vh)) * e.vol / e.v.numel()}
