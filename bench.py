"""Benchmark: H|psi> state-applies per second on the Si64 configuration.

One step = one application of H to the whole 128-state block of the 64-atom
Si supercell (L = 20.52 bohr, 72^3 grid, E_cut = 30 Ha, Gamma, 64 Gaussian
s+p KB projectors), states resident in HBM on their G sphere.  The headline
value is the mixed-precision (complex64) path; the FP64 path is timed on the
same input and reported beside it, with the FP32-vs-FP64 error on H|psi> and
on the band energy per atom.  The dominant kernel's achieved HBM bandwidth
comes from HIP events recorded around each launch on the library's stream.

Secondary lines in the same JSON object (same seeded inputs):
  hbm_copy      plain streaming copy kernel, the measured HBM reference
  c3_kpoints    Al4 fcc, 64 k-points x 2 spins (128 uneven blocks, each spin reading its own
                potential component) in one batched launch
  c4_tddft      ETRS steps on Si64 with a velocity-gauge kick, hipGraph replay,
                FP32 vs FP64 dipole trace and energy drift
  c1_diamond    C8 diamond apply + overlap + Cholesky, GPU and CPU oracle
  c5_ace        Si216 (96^3, 432 states) ACE build: all pair-density Poisson solves,
                W^H phi, FP64 Cholesky, xi; ACE apply; FP32 vs FP64 direct exchange
  contractions  overlap and rotate on the matrix cores at the Si64 and Si216 block
                sizes, TFLOP/s and fraction of the dense MFMA peak; FP64 Cholesky and L^-1
  sd_si64       steepest_descent (5 preconditioned steps + orthogonalize) on the Si64 block
  scf_steps     Si216 ionic density (216 atomic spheres) and Hartree solve at 96^3;
                restart save/load of 32 Si64 states
The CPU baseline is the FP64 oracle (a C/OpenMP port of the reference CPU data
flow) on a bounded subset of the Si64 states.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--precision fp32|fp64|both]
                       [--no-cpu] [--no-extras]
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
METRIC = "state-applies of H/sec + HBM GB/s; FP32-mixed vs FP64 at <=1e-6 Ha/atom"


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def cpu_threads():
    """threads of the CPU baseline: OMP_NUM_THREADS when set, else the cores this
    process may run on"""
    n = int(os.environ.get("OMP_NUM_THREADS", "0") or 0)
    if n > 0:
        return n
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:
        return os.cpu_count() or 1


def cpu_host():
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {"cpu_model": model, "nproc": os.cpu_count(), "threads_used": cpu_threads()}


def median_time(fn, warmup=3, reps=10, min_seconds=0.0):
    """3 warm-ups, then the median of at least `reps` timed calls (more while
    the total stays under min_seconds)"""
    for _ in range(warmup):
        fn()
    ts = []
    t_start = time.perf_counter()
    while len(ts) < reps or time.perf_counter() - t_start < min_seconds:
        t0 = time.perf_counter()
        fn()
        ts.append(time.perf_counter() - t0)
        if len(ts) >= 200:
            break
    return float(np.median(ts)), len(ts)


def kernel_bytes(name, nst, npw, nslot, n12, N, prec_bytes):
    """algorithmic HBM bytes of one launch of a pipeline kernel on nst states:
    compulsory reads + writes of the streams it touches (the plane
    intermediates hold nslot planes of n12 points per state)."""
    cs = 2 * prec_bytes
    plane = nslot * n12 * cs
    if name.startswith("plane_inverse"):
        return nst * (npw * cs + plane)
    if name.startswith("xpass_project"):
        return nst * plane
    if name.startswith("xpass_apply"):
        return nst * 2 * plane + N * prec_bytes
    if name.startswith("plane_forward"):
        return nst * (plane + 2 * npw * cs)
    return 0


COUNTER_PROFILE = os.path.join(ROOT, "profiles", "hpsi_si64_fp32_hbm_counters.txt")


def counter_traffic(kernel):
    """HBM bytes per launch of a complex64 Si64 pipeline kernel, from the committed
    FETCH_SIZE/WRITE_SIZE counter passes (already scaled by the copy-kernel
    calibration: 2 x FETCH + 1 x WRITE).  None when the kernel has no row."""
    stem = kernel.rsplit("_f", 1)[0]
    try:
        with open(COUNTER_PROFILE) as f:
            for line in f:
                parts = line.split()
                if len(parts) >= 5 and parts[0].startswith("k_" + stem + "<"):
                    return float(parts[4]) * 2**20
    except OSError:
        return None
    return None


def b_alg(npw, N, nsph, nst, s_c, s_r, nlm=4):
    """algorithmic bytes per state-apply of the 2-pass FFT model:
    s_c (2 N_pw + 4 N + 3 N_sph) + [s_r N + N_sph (nlm s_r + 24)] / nst"""
    return s_c * (2 * npw + 4 * N + 3 * nsph) + (s_r * N + nsph * (nlm * s_r + 24)) / nst


def build(ctx, sysm, v=None):
    from inq_amd import KSHamiltonian
    from inq_amd import systems as S
    gh = KSHamiltonian(ctx, sysm.lattice, sysm.n)
    gh.set_scalar_potential(S.local_potential(sysm) if v is None else v)
    for p, D in zip(sysm.positions, sysm.kb_coeffs()):
        gh.add_projector(p, sysm.kb_radius, sysm.nlm, D, width=sysm.kb_width)
    return gh


def time_applies(ctx, gh, b, d_in, d_out, steps, warmup):
    for _ in range(warmup):
        gh.apply(b, d_in, d_out)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(steps):
        gh.apply(b, d_in, d_out)
    ctx.sync()
    return (time.perf_counter() - t0) / steps


def hbm_copy(ctx, nbytes=1 << 31, reps=10):
    from inq_amd import DeviceArray, lib
    a = DeviceArray(ctx, (nbytes // 8,), np.complex64)
    b = DeviceArray(ctx, (nbytes // 8,), np.complex64)
    for _ in range(2):
        lib().inqx_stream_copy(ctx.h, a.ptr, b.ptr, nbytes)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(reps):
        lib().inqx_stream_copy(ctx.h, a.ptr, b.ptr, nbytes)
    ctx.sync()
    dt = (time.perf_counter() - t0) / reps
    a.free()
    b.free()
    return 2 * nbytes / dt / 1e9


def tune_cache():
    """the autotuner's cache file: INQX_TUNE_CACHE, else ~/.cache/inqx/tune.txt"""
    path = os.environ.get("INQX_TUNE_CACHE") or os.path.join(os.path.expanduser("~"), ".cache", "inqx", "tune.txt")
    try:
        os.makedirs(os.path.dirname(path), exist_ok=True)
    except OSError:
        return None
    return path


def c3_kpoints(ctx, steps):
    from inq_amd import DeviceArray
    from inq_amd import systems as S
    sysm = S.config(3)
    gh = build(ctx, sysm)
    # spin-polarised: a two-component potential [N][2], each block reading its spin's
    v = S.local_potential(sysm)
    gh.set_scalar_potential(np.stack([v, v + 0.3 * np.random.default_rng(5).standard_normal(v.shape)], axis=1), ncomp=2)
    vol = S.sphere_volume_element(sysm)
    bases, ins, outs = [], [], []
    for i, (k, spin, ec) in enumerate(sysm.blocks()):
        b = gh.basis(k, ec, spin)
        c = S.random_states(b.npw, sysm.nst, sysm.seed + i, vol).astype(np.complex64)
        bases.append(b)
        ins.append(DeviceArray.from_numpy(ctx, c))
        outs.append(DeviceArray(ctx, c.shape, np.complex64))
    npws = [b.npw for b in bases]
    t0 = time.perf_counter()
    shape, tuned_ms = gh.autotune_batch(bases, [sysm.nst] * len(bases), np.complex64, tune_cache())
    t_tune = time.perf_counter() - t0
    gh.apply_batch(bases, ins, outs)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(steps):
        gh.apply_batch(bases, ins, outs)
    ctx.sync()
    dt = (time.perf_counter() - t0) / steps
    nsa = sysm.nst * len(bases)
    return {"blocks": len(bases), "spins": sorted({int(b.spin) for b in bases}), "nst": sysm.nst,
            "npw_min": int(min(npws)), "npw_max": int(max(npws)),
            "ms_per_batch": dt * 1e3, "state_applies_per_s": nsa / dt, "dtype": "c64",
            "launch_shape": {"xpass_states_per_wg": shape[0], "planes_per_wg": shape[1], "tune_s": t_tune}}


def c4_tddft(ctx, nsteps):
    from inq_amd import DeviceArray
    from inq_amd import real_time as rt
    from inq_amd import systems as S
    sysm = S.config(4)
    v = S.local_potential(sysm)
    out = {}
    recs = {}
    for dtype, name in ((np.complex64, "fp32"), (np.complex64, "fp32_fp64state"), (np.complex128, "fp64")):
        gh = build(ctx, sysm, v)
        # velocity-gauge kick 0.01 along x: A = -0.01 x (src/perturbations/kick.hpp:36-48), covariant
        gh.uniform_vector_potential = sysm.lattice @ np.array([-0.01, 0.0, 0.0])
        b = gh.basis((0, 0, 0), sysm.ecut)
        c = S.random_states(b.npw, sysm.nst, sysm.seed, S.sphere_volume_element(sysm))
        d = DeviceArray.from_numpy(ctx, c.astype(dtype))
        prop = rt.Propagator(gh, [b], [d], [np.full(sysm.nst, 2.0)], dt=0.05, ring_capacity=nsteps + 8)
        if name == "fp32_fp64state":
            prop.set_state_precision(np.complex128)  # FP32 applications, complex128 states
        prop.energy()
        prop.step(2, graph=True)  # eager first step + capture
        ctx.sync()
        t0 = time.perf_counter()
        prop.step(nsteps, graph=True)
        ctx.sync()
        dt = (time.perf_counter() - t0) / nsteps
        recs[name] = prop.records(cap=nsteps + 8)
        out[name] = {"ms_per_step": dt * 1e3, "steps_per_s": 1.0 / dt,
                     "state_applies_per_s": 9 * sysm.nst / dt}
        prop.close()
        del prop
    r32, r64, rw = recs["fp32"], recs["fp64"], recs["fp32_fp64state"]
    m = min(len(r32), len(r64), len(rw))
    out["fp32_fp64state_band_energy_err_per_atom_Ha"] = float(np.max(np.abs(rw[:m, 1] - r64[:m, 1])) / sysm.natoms)
    out["fp32_fp64state_dipole_trace_max_abs_err"] = float(np.max(np.abs(rw[:m, 4:7] - r64[:m, 4:7])))
    out["fp32_fp64state_norm_vs_fp64"] = float(np.max(np.abs(rw[:m, 3] - r64[:m, 3])) / sysm.nst)
    dip_err = float(np.max(np.abs(r32[:m, 4:7] - r64[:m, 4:7])))
    e32 = r32[:m, 1]
    e64 = r64[:m, 1]
    out["steps"] = int(m - 1)
    out["dipole_trace_max_abs_err_fp32_vs_fp64"] = dip_err
    out["dipole_trace_max_abs"] = float(np.max(np.abs(r64[:m, 4:7])))
    # the seeded states fill the whole sphere up to 30 Ha, where the Taylor-4
    # step (dt/2 * 30 Ha = 0.75) is slightly dissipative: the drift is the
    # propagator's (identical in FP32 and FP64), the FP32-vs-FP64 gap is precision
    out["energy_drift_fp64_rel"] = float(abs(e64[-1] - e64[0]) / abs(e64[0]))
    out["energy_drift_fp32_rel"] = float(abs(e32[-1] - e32[0]) / abs(e32[0]))
    out["band_energy_err_per_atom_Ha"] = float(np.max(np.abs(e32 - e64)) / sysm.natoms)
    out["norm_drift_fp64"] = float(np.max(np.abs(r64[:m, 3] - sysm.nst)) / sysm.nst)
    out["norm_fp32_vs_fp64"] = float(np.max(np.abs(r32[:m, 3] - r64[:m, 3])) / sysm.nst)
    return out


def c1_diamond(ctx, cpu):
    from inq_amd import DeviceArray
    from inq_amd import operations as ops
    from inq_amd import systems as S
    sysm = S.config(1)
    v = S.local_potential(sysm)
    gh = build(ctx, sysm, v)
    b = gh.basis((0, 0, 0), sysm.ecut)
    vol = S.sphere_volume_element(sysm)
    c = S.random_states(b.npw, sysm.nst, sysm.seed, vol)
    d = DeviceArray.from_numpy(ctx, c)
    h = DeviceArray(ctx, c.shape, np.complex128)

    def gpu_once():
        gh.apply(b, d, h)
        S_ = ops.overlap(ctx, d, d, vol)
        ops.cholesky(ctx, S_)

    gpu_once()
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(20):
        gpu_once()
    ctx.sync()
    res = {"gpu_fp64_ms": (time.perf_counter() - t0) / 20 * 1e3}
    if cpu:
        from oracle import oracle as orc
        oh = orc.Ham(sysm.lattice, sysm.n)
        oh.set_potential(v)
        for p, D in zip(sysm.positions, sysm.kb_coeffs()):
            oh.add_projector_gauss(p, sysm.kb_radius, sysm.nlm, sysm.kb_width, D)
        g = b.gindex()
        threads = cpu_threads()
        rc = orc.RefCPU(oh, sysm.nst, threads)
        cube = np.zeros((sysm.N, sysm.nst), dtype=np.complex128)
        cube[g] = c.T
        hc = np.zeros_like(cube)

        def cpu_once():
            rc.apply(cube, hc)
            orc.ref_overlap_cholesky(cube, vol)

        t_med, reps = median_time(cpu_once, 3, 10, 2.0)
        res["cpu_fp64_ms"] = t_med * 1e3
        res["cpu"] = {"backend": rc.backend, "threads": threads, "reps": reps, "statistic": "median after 3 warm-ups",
                      "path": "full-cube [x][y][z][ist] apply (batched FFTW3, DGEMM KB) + ZGEMM overlap + ZPOTRF"}
        res["gpu_vs_cpu"] = res["cpu_fp64_ms"] / res["gpu_fp64_ms"]
    return res


MFMA_PEAK_TFLOPS = {"fp32": 157.3, "fp64": 78.6}  # MI355X dense matrix-core peaks


def contractions(ctx, reps=10):
    """The dense contractions on the matrix cores: the overlap S = vol phi^H phi
    (operations::overlap) and the rotation phi R (operations::rotate) at the
    Si64 block (128 x 67 691) and the Si216 block (432 x 228 487).  8 n^2 K flop
    for the rotation (complex multiply-add), 4 n (n + 1) K for the overlap of a
    block with itself (Hermitian: its lower triangle), timed per kernel with the
    library's HIP events;
    utilisation is against the dense FP32 / FP64 MFMA peak."""
    from inq_amd import DeviceArray
    from inq_amd import operations as ops
    out = {}
    rng = np.random.default_rng(3)
    for name, n, K in (("si64", 128, 67691), ("si216", 432, 228487)):
        for dtype, prec in ((np.complex64, "fp32"), (np.complex128, "fp64")):
            a = (rng.standard_normal((n, K)) + 1j * rng.standard_normal((n, K))).astype(dtype)
            d = DeviceArray.from_numpy(ctx, a)
            rot = DeviceArray.from_numpy(ctx, np.eye(n, dtype=np.complex128))
            ops.overlap(ctx, d, d, 1.0).free()
            ops.rotate(ctx, rot, d)
            ctx.sync()
            ctx.profile(True)
            ctx.profile_reset()
            for _ in range(reps):
                ops.overlap(ctx, d, d, 1.0).free()
                ops.rotate(ctx, rot, d)
            kt = ctx.kernel_times()
            ctx.profile(False)
            flops = {"overlap": 4.0 * n * (n + 1) * K, "rotate": 8.0 * n * n * K}
            res = {}
            sfx = "f32" if prec == "fp32" else "f64"
            for kind, key in (("overlap", f"overlap_mfma_{sfx}"), ("rotate", f"rotate_mfma_{sfx}")):
                cnt, ms = kt[key]
                tf = flops[kind] / (ms / cnt * 1e-3) / 1e12
                res[kind] = {"us": ms / cnt * 1e3, "tflops": tf, "frac_of_mfma_peak": tf / MFMA_PEAK_TFLOPS[prec]}
            cnt, ms = kt[f"overlap_reduce_{sfx}"]
            res["overlap"]["reduce_us"] = ms / cnt * 1e3
            out[f"{name}_{prec}"] = res
            d.free()
            rot.free()
        # the FP64 steps between overlap and rotate in orthogonalize: Cholesky and L^-1
        s = a[:, :n].astype(np.complex128)
        s = s @ s.conj().T + n * np.eye(n)
        lmat = DeviceArray.from_numpy(ctx, np.linalg.cholesky(s))
        ops.invert_triangular(ctx, lmat).free()
        ctx.sync()
        ctx.profile(True)
        ctx.profile_reset()
        for _ in range(reps):
            ops.cholesky(ctx, DeviceArray.from_numpy(ctx, s)).free()
            ops.invert_triangular(ctx, lmat).free()
        kt = ctx.kernel_times()
        ctx.profile(False)
        out[f"{name}_fp64"]["cholesky_us"] = kt["cholesky_f64"][1] / kt["cholesky_f64"][0] * 1e3
        out[f"{name}_fp64"]["trinv_us"] = kt["trinv_f64"][1] / kt["trinv_f64"][0] * 1e3
        lmat.free()
    return out


def sd_si64(ctx, gh, b, c, nst, reps=5):
    """One ground-state eigensolver step of the Si64 block: steepest_descent(ham,
    prec, phi) with 5 preconditioned line minimisations per state and the closing
    orthogonalisation (src/eigensolvers/steepest_descent.hpp:23-86, called with
    these arguments from src/ground_state/calculator.hpp:160-168).  Timed per call
    around a device synchronisation; the kernel split comes from the library's HIP
    events in a separate pass."""
    from inq_amd import DeviceArray
    from inq_amd import eigensolvers as es
    out = {}
    for dtype, prec in ((np.complex64, "fp32"), (np.complex128, "fp64")):
        d = DeviceArray.from_numpy(ctx, c.astype(dtype))
        gh.prepare(b, nst, dtype)
        es.steepest_descent(gh, b, d)
        ctx.sync()
        t0 = time.perf_counter()
        for _ in range(reps):
            es.steepest_descent(gh, b, d)
        ctx.sync()
        dt = (time.perf_counter() - t0) / reps
        ctx.profile(True)
        ctx.profile_reset()
        es.steepest_descent(gh, b, d)
        kt = ctx.kernel_times()
        ctx.profile(False)
        groups = {"h_apply": ("plane_", "xpass_", "kb_reduce"), "sd_vector_ops": ("sd_", "tpa_", "precondition"),
                  "orthogonalize": ("overlap_", "cholesky", "trinv", "rotate_")}
        split = {g: sum(ms for k, (cnt, ms) in kt.items() if k.startswith(pre)) for g, pre in groups.items()}
        out[prec] = {"ms_per_call": dt * 1e3, "states_per_s": nst / dt,
                     "kernel_ms": {g: v for g, v in split.items()},
                     "kernel_ms_other": sum(ms for _, ms in kt.values()) - sum(split.values())}
        d.free()
    return out


def scf_steps(ctx, gh64, b64, c64, reps=5):
    """The steps around H in a self-consistent run, on the device:
    ionic density of Si216 (216 atoms, 96^3, atomic_potential::ionic_density,
    atomic_potential.hpp:170-200, declared Gaussian of width 0.625) and its
    Hartree potential and energy (self_consistency.hpp:115-120), plus a restart
    round trip of 32 Si64 states (io::save / io::load, io.hpp:168-211: one
    complex128 real-space file per state) through a temporary directory."""
    import shutil
    import tempfile
    from inq_amd import DeviceArray, KSHamiltonian
    from inq_amd import io as inqio
    from inq_amd import potential as pot
    from inq_amd import systems as S
    out = {}
    sysm = S.config(5)
    gh = KSHamiltonian(ctx, sysm.lattice, sysm.n)
    z = np.full(sysm.natoms, 4.0)
    rho = pot.ionic_density(gh, sysm.positions, z)
    vh, eh = gh.hartree(rho)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(reps):
        rho.upload(np.zeros(sysm.N))
        pot.ionic_density(gh, sysm.positions, z, field=rho)
    ctx.sync()
    t_rho = (time.perf_counter() - t0) / reps
    t0 = time.perf_counter()
    for _ in range(reps):
        gh.hartree(rho, vh)
    ctx.sync()
    t_h = (time.perf_counter() - t0) / reps
    dv = abs(np.linalg.det(sysm.lattice)) / sysm.N
    out["si216_ionic_density_ms"] = t_rho * 1e3
    out["si216_ionic_charge"] = float(rho.numpy().sum() * dv)
    out["si216_hartree_ms"] = t_h * 1e3
    out["si216_hartree_energy_Ha"] = eh
    rho.free()
    vh.free()
    nst = 32
    d = DeviceArray.from_numpy(ctx, c64[:nst].astype(np.complex64))
    back = DeviceArray(ctx, d.shape, np.complex64)
    tmp = tempfile.mkdtemp(prefix="inqx_restart_")
    try:
        t0 = time.perf_counter()
        inqio.save_states(gh64, b64, d, os.path.join(tmp, "states"))
        t_save = time.perf_counter() - t0
        t0 = time.perf_counter()
        inqio.load_states(gh64, b64, back, os.path.join(tmp, "states"))
        ctx.sync()
        t_load = time.perf_counter() - t0
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    nbytes = 16 * nst * int(np.prod(gh64.n))
    a, bb = d.numpy(), back.numpy()
    out["restart_states"] = nst
    out["restart_bytes"] = nbytes
    out["restart_save_gbs"] = nbytes / t_save / 1e9
    out["restart_load_gbs"] = nbytes / t_load / 1e9
    out["restart_round_trip_rel"] = float(np.max(np.abs(bb - a)) / np.max(np.abs(a)))
    d.free()
    back.free()
    return out


def c5_ace(ctx, cpu, cpu_seconds=8.0):
    """ACE build on Si216 (96^3, 432 complex64 states, Gamma): nst^2 pair-density
    Poisson solves + W^H phi + FP64 Cholesky + xi = W L^-H, and one ACE apply."""
    from inq_amd import DeviceArray, KSHamiltonian
    from inq_amd import operations as ops
    from inq_amd import systems as S
    from inq_amd.exchange import ExchangeOperator
    sysm = S.config(5)
    gh = KSHamiltonian(ctx, sysm.lattice, sysm.n)
    b = gh.basis((0, 0, 0), sysm.ecut)
    nst, N = sysm.nst, sysm.N
    vol = S.sphere_volume_element(sysm)
    rng = np.random.default_rng(sysm.seed)
    c = rng.standard_normal((nst, b.npw)) + 1j * rng.standard_normal((nst, b.npw))
    d64 = DeviceArray.from_numpy(ctx, c)
    ops.orthogonalize(ctx, d64, vol)  # FP64 Cholesky orthonormalisation on the device
    c = d64.numpy()
    d = DeviceArray.from_numpy(ctx, c.astype(np.complex64))
    occ = np.full(nst, 2.0)
    ex = ExchangeOperator(gh, b, exchange_coefficient=1.0)
    ex.update(d, occ)  # warm-up: workspaces and descriptors
    ctx.sync()
    ctx.profile(True)
    ctx.profile_reset()
    t0 = time.perf_counter()
    energy = ex.update(d, occ)
    ctx.sync()
    t_build = time.perf_counter() - t0
    kt = ctx.kernel_times()
    ctx.profile(False)
    out = DeviceArray(ctx, c.shape, np.complex64)
    out.upload(np.zeros(c.shape, np.complex64))
    ex.ace(d, out)
    ctx.sync()
    t0 = time.perf_counter()
    for _ in range(5):
        ex.ace(d, out)
    ctx.sync()
    t_apply = (time.perf_counter() - t0) / 5
    pairs = nst * nst
    # every state is occupied and the pair potentials of (i, j) and (j, i) are
    # complex conjugates: the build solves each unordered pair once
    solved = nst * (nst + 1) // 2
    sc = 8
    # per solved pair: phi_i read and t written (plane_fwd), t read+written (xline), t
    # read+written (plane_inv), t read (reduce); per conjugate pair one t read
    # (reduce_sym); hf_j is shared by all i and w_i is amortised over the chunk
    pair_bytes = 7 * N * sc
    build_bytes = solved * pair_bytes + (pairs - solved) * N * sc
    kern = {k: v[1] / v[0] * 1e3 for k, v in kt.items()}
    pk = {k: kern[k] for k in kern if k.startswith("pair_")}
    res = {"states": nst, "grid": list(sysm.n), "npw": int(b.npw), "pairs": pairs, "pairs_solved": solved,
           "build_s": t_build, "pair_solves_per_s": pairs / t_build,
           "poisson_solves_per_s": solved / t_build,
           "exchange_energy_Ha": energy, "ace_apply_ms": t_apply * 1e3,
           "pair_bytes": pair_bytes,
           "pair_pipeline_gbs": build_bytes / (sum(kt[k][1] for k in kt if k.startswith("pair_")) * 1e-3) / 1e9,
           "kernels_us": pk}
    # complex64 direct exchange of all states with 4 occupied states, twice (the
    # repeats must agree bit for bit: fixed reduction orders); the first 8 outputs
    # are checked against the FP64 oracle below (complex128 exchange is not offered
    # above 64^3)
    hf_idx = 4
    d32h = DeviceArray.from_numpy(ctx, c[:hf_idx].astype(np.complex64))
    k32 = [ex.direct(d, d32h, occ[:hf_idx]).numpy().astype(np.complex128) for _ in range(2)]
    scale32 = np.max(np.abs(k32[0]))
    res["direct_repeat_rel_fp32"] = float(np.max(np.abs(k32[1] - k32[0])) / scale32)
    for a in (d32h, out, d, d64):
        a.free()
    if cpu:
        # CPU leg: the FP64 oracle checks 8 outputs, and the reference CPU path is timed
        from oracle import oracle as orc
        ns = 8
        oh = orc.Ham(sysm.lattice, sysm.n)
        ng = tuple(sysm.n)
        g = b.gindex()
        cube = np.zeros((ns, N), dtype=np.complex128)
        cube[:, g] = c[:ns].astype(np.complex64)
        rs_all = np.fft.ifftn(cube.reshape((ns,) + ng), axes=(1, 2, 3)).reshape(ns, N)
        kr = oh.exchange_direct(np.ascontiguousarray(rs_all.T), np.ascontiguousarray(rs_all[:hf_idx].T),
                                occ[:hf_idx], exx_coeff=1.0, scale=1.0)
        kref = np.fft.fftn(np.ascontiguousarray(kr.T).reshape((ns,) + ng), axes=(1, 2, 3)).reshape(ns, N)[:, g]
        res["direct_fp32_vs_fp64_oracle_rel"] = float(np.max(np.abs(k32[0][:ns] - kref)) / np.max(np.abs(kref)))
        res["direct_check"] = f"{ns} of {nst} states x {hf_idx} occupied states against the FP64 oracle"
        threads = cpu_threads()
        nsc = max(ns, threads)  # one state per thread at least
        cube = np.zeros((nsc, N), dtype=np.complex128)
        cube[:, g] = c[:nsc]
        rs = np.fft.ifftn(cube.reshape((nsc,) + ng), axes=(1, 2, 3)).reshape(nsc, N)
        rs = np.ascontiguousarray(rs.T)  # [N][nsc], the reference's point-major layout
        hf = np.ascontiguousarray(rs[:, :1])
        coef = np.array([-0.5 * occ[0]])
        t_med, reps = median_time(lambda: orc.ref_exchange_pairs(sysm.lattice, sysm.n, rs, hf, coef, threads),
                                  3, 10, 0.0)
        res["cpu_reference_path"] = {
            "pair_solves_per_s": nsc / t_med, "threads": threads, "reps": reps,
            "statistic": "median after 3 warm-ups",
            "sample": f"{nsc} states x 1 occupied state, FP64 pair solves at 96^3 (batched FFTW3 over states)"}
        res["gpu_vs_cpu_pair_solves"] = res["pair_solves_per_s"] / (nsc / t_med)
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--precision", default="both", choices=("fp32", "fp64", "both"))
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extras", action="store_true")
    ap.add_argument("--copy", action="store_true", help="run the HBM copy reference even with --no-extras")
    ap.add_argument("--only-c5", action="store_true", help="run only the Si216 ACE line (profiling)")
    ap.add_argument("--only-contractions", action="store_true", help="run only the overlap / rotate timing")
    ap.add_argument("--only-sd", action="store_true", help="run only the Si64 steepest-descent line")
    ap.add_argument("--only-scf-steps", action="store_true", help="run only the ionic density / Hartree / restart line")
    ap.add_argument("--only-c4", action="store_true", help="run only the Si64 TDDFT line (profiling)")
    ap.add_argument("--c4-steps", type=int, default=2000, help="ETRS steps of the Si64 TDDFT line")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {args.gpus}); "
              "the multi-GPU sharding of the path is design only and not measured.", file=sys.stderr)
        sys.exit(2)

    from inq_amd import Context, DeviceArray
    from inq_amd import systems as S

    if args.only_c5:
        res = c5_ace(Context(0), not args.no_cpu)
        print(json.dumps({"c5_ace": res}), flush=True)
        return
    if args.only_contractions:
        print(json.dumps({"contractions": contractions(Context(0))}), flush=True)
        return
    if args.only_c4:
        print(json.dumps({"c4_tddft": c4_tddft(Context(0), args.c4_steps)}), flush=True)
        return

    sysm = S.config(2)
    log(f"bench: {sysm.name}, {sysm.natoms} atoms, nst={sysm.nst}")
    v = S.local_potential(sysm)
    ctx = Context(0)
    gh = build(ctx, sysm, v)
    b = gh.basis((0, 0, 0), sysm.ecut)
    vol = S.sphere_volume_element(sysm)
    c = S.random_states(b.npw, sysm.nst, sysm.seed, vol)
    gidx = b.gindex()
    nslot = len(np.unique(gidx // (sysm.n[1] * sysm.n[2])))
    n12 = sysm.n[1] * sysm.n[2]
    nsph = sum(len(gh.projector_points(a)[0]) for a in range(sysm.natoms))

    if args.only_sd:
        print(json.dumps({"sd_si64": sd_si64(ctx, gh, b, c, sysm.nst)}), flush=True)
        return
    if args.only_scf_steps:
        print(json.dumps({"scf_steps": scf_steps(ctx, gh, b, c)}), flush=True)
        return

    res, outs = {}, {}
    precs = {"fp32": [np.complex64], "fp64": [np.complex128], "both": [np.complex64, np.complex128]}[args.precision]
    for dtype in precs:
        name = "fp32" if dtype == np.complex64 else "fp64"
        d_in = DeviceArray.from_numpy(ctx, c.astype(dtype))
        d_out = DeviceArray(ctx, c.shape, dtype)
        gh.prepare(b, sysm.nst, dtype)
        shape, _ = gh.autotune_batch([b], [sysm.nst], dtype, tune_cache())
        dt = time_applies(ctx, gh, b, d_in, d_out, args.steps, args.warmup)
        ctx.profile(True)
        ctx.profile_reset()
        for _ in range(args.steps):
            gh.apply(b, d_in, d_out)
        ktimes = ctx.kernel_times()
        ctx.profile(False)
        outs[name] = d_out.numpy().astype(np.complex128)
        res[name] = {"ms": dt * 1e3, "rate": sysm.nst / dt, "kernels": ktimes,
                     "launch_shape": {"xpass_states_per_wg": shape[0], "planes_per_wg": shape[1]}}
        log(f"bench: {name} {dt * 1e3:.3f} ms per {sysm.nst}-state apply, {sysm.nst / dt:.4g} state-applies/s")
        for kname, (cnt, ms) in sorted(ktimes.items()):
            log(f"   {kname:24s} {ms / cnt * 1e3:9.1f} us/launch")
        d_in.free()
        d_out.free()

    head = "fp32" if "fp32" in res else "fp64"
    prec_bytes = 4 if head == "fp32" else 8
    kt = res[head]["kernels"]
    dom = max(kt, key=lambda k: kt[k][1])
    cnt, ms = kt[dom]
    avg_s = ms / cnt * 1e-3
    kb = kernel_bytes(dom, sysm.nst, b.npw, nslot, n12, sysm.N, prec_bytes)
    achieved = kb / avg_s / 1e9
    rate = res[head]["rate"]
    balg = b_alg(b.npw, sysm.N, nsph, sysm.nst, 2 * prec_bytes, prec_bytes)

    out = {
        "metric": METRIC,
        "value": rate,
        "unit": "state-applies/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": res[head]["ms"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64 (f32)" if head == "fp32" else "c128 (f64)",
        "data": "synthetic (seeded N(0,1) states on the G sphere, Gaussian V_loc and KB projectors)",
        "config": {"workload": "H|psi> on Si64 2x2x2 diamond, L=20.52 bohr, 72^3 grid, Ecut 30 Ha, Gamma, "
                               "128 states, 64 atoms x 4 KB projectors (r_c 2.0)",
                   "npw": int(b.npw), "n_sph": int(nsph), "nst": sysm.nst, "grid": list(sysm.n)},
        "hbm_gbs_effective_b_alg": balg * rate / 1e9,
        "b_alg_bytes_per_state_apply": balg,
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS,
                     "traffic": counter_traffic(dom) if head == "fp32" else None,
                     "traffic_source": "profiles/hpsi_si64_fp32_hbm_counters.txt (2 x FETCH_SIZE + WRITE_SIZE)",
                     "bytes_per_launch": kb, "avg_launch_us": avg_s * 1e6},
        "kernels_us": {k: vv[1] / vv[0] * 1e3 for k, vv in kt.items()},
        "launch_shape": res[head]["launch_shape"],
    }
    if "fp32" in res and "fp64" in res:
        ci = c.astype(np.complex64).astype(np.complex128)
        h32, h64 = outs["fp32"], outs["fp64"]
        e32 = np.real(np.sum(ci.conj() * h32, 1)) * vol
        e64 = np.real(np.sum(ci.conj() * h64, 1)) * vol
        out["fp64"] = {"value": res["fp64"]["rate"], "ms_per_step": res["fp64"]["ms"],
                       "kernels_us": {k: vv[1] / vv[0] * 1e3 for k, vv in res["fp64"]["kernels"].items()}}
        out["speedup_fp32_vs_fp64"] = res["fp32"]["rate"] / res["fp64"]["rate"]
        out["err_fp32_vs_fp64"] = {"hpsi_rel_max": float(np.max(np.abs(h32 - h64)) / np.max(np.abs(h64))),
                                   "band_energy_per_atom_Ha": float(abs(np.sum(e32) - np.sum(e64)) / sysm.natoms)}

    if args.copy and args.no_extras:
        out["hbm_copy_gbs"] = hbm_copy(ctx)
    if not args.no_extras:
        out["hbm_copy_gbs"] = hbm_copy(ctx)
        log(f"bench: hbm copy {out['hbm_copy_gbs']:.0f} GB/s")
        out["c3_kpoints"] = c3_kpoints(ctx, max(3, args.steps // 4))
        log(f"bench: c3 {out['c3_kpoints']}")
        out["c4_tddft"] = c4_tddft(ctx, args.c4_steps)
        log(f"bench: c4 {out['c4_tddft']}")
        out["c1_diamond"] = c1_diamond(ctx, not args.no_cpu)
        log(f"bench: c1 {out['c1_diamond']}")
        out["c5_ace"] = c5_ace(ctx, not args.no_cpu)
        log(f"bench: c5 {out['c5_ace']}")
        out["contractions"] = contractions(ctx)
        log(f"bench: contractions {out['contractions']}")
        out["sd_si64"] = sd_si64(ctx, gh, b, c, sysm.nst)
        log(f"bench: sd {out['sd_si64']}")
        out["scf_steps"] = scf_steps(ctx, gh, b, c)
        log(f"bench: scf steps {out['scf_steps']}")

    cpu = None
    if not args.no_cpu:
        from oracle import oracle as orc
        threads = cpu_threads()
        oh = orc.Ham(sysm.lattice, sysm.n)
        oh.set_potential(v)
        for p, D in zip(sysm.positions, sysm.kb_coeffs()):
            oh.add_projector_gauss(p, sysm.kb_radius, sysm.nlm, sysm.kb_width, D)
        nsub = 32
        rc = orc.RefCPU(oh, nsub, threads)
        cube = np.zeros((sysm.N, nsub), dtype=np.complex128)
        cube[gidx] = c[:nsub].T
        hc = np.zeros_like(cube)
        t_med, reps = median_time(lambda: rc.apply(cube, hc), 3, 10, args.cpu_seconds)
        # the reference CPU path agrees with the FP64 GPU apply on the same states
        if "fp64" in outs:
            ref_err = float(np.max(np.abs(hc[gidx].T - outs["fp64"][:nsub])) / np.max(np.abs(outs["fp64"][:nsub])))
        else:
            ref_err = None
        host = cpu_host()
        cpu = {"value": nsub / t_med, "unit": "state-applies/s", "cores": threads, "kind": "port",
               "backend": rc.backend, "statistic": f"median of {reps} after 3 warm-ups",
               "cpu_model": host["cpu_model"], "nproc": host["nproc"],
               "gpu_fp64_vs_cpu_rel_err": ref_err,
               "sample": f"H on {nsub} of the {sysm.nst} Si64 states as the reference's CPU path runs it: full 72^3 "
                         f"cube [x][y][z][ist] in Fourier space, batched FFTW3 transforms over states "
                         f"(MKL's FFTW3 interface, sequential per thread), x 1/N pass, V psi, KB by DGEMM on "
                         f"interleaved re/im, FP64, {threads} OpenMP threads over state chunks"}
        log(f"bench: cpu reference path {nsub / t_med:.4g} state-applies/s on {threads} threads ({rc.backend})")
    out["cpu_baseline"] = cpu
    print(json.dumps(out))


if __name__ == "__main__":
    main()
