"""GPU parity of H on grids whose whole cube fits one work-group's LDS (one
launch, a work-group per state) against the FP64 oracle: the smallest and the
largest cubes, three different axes, k != 0, overlapping projector spheres,
d channels (several groups per projector), no projectors, batches of uneven
blocks, Taylor accumulators, and the grids just above the limit, which take the
plane passes.

Tolerances as in test_gpu_hamiltonian.py: 1e-11 complex128, 2e-5 complex64."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, KSHamiltonian
from inq_amd import real_time as rt
from inq_amd import systems as S
from oracle import oracle as orc
from tests.helpers import gpu_ham, oracle_ham, rel_err, say

pytestmark = pytest.mark.gpu

TOL = {np.complex128: 1e-11, np.complex64: 2e-5}
DTYPES = [np.complex128, np.complex64]


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


def _system(n, natoms, nst=3, seed=0):
    rng = np.random.default_rng(sum(n) + seed)
    L = np.diag([0.28 * x for x in n])
    return S.System("cube", 400 + sum(n), L, n, rng.uniform(-0.5, 0.5, (natoms, 3)) @ L, 18.0, nst,
                    v_sigma=0.6, kb_width=0.7, kb_radius=1.6)


GRIDS = [(12, 12, 12), (16, 16, 16), (18, 16, 20), (20, 20, 20), (24, 20, 18), (24, 24, 24), (30, 16, 24), (12, 32, 20),
         (28, 20, 20), (24, 24, 30)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", GRIDS)
@pytest.mark.parametrize("k", [(0.0, 0.0, 0.0), (0.3, -0.2, 0.45)])
def test_h(ctx, dtype, n, k):
    say("case: small cube", n, k, np.dtype(dtype).name)
    sysm = _system(n, 5)
    gh, oh = gpu_ham(ctx, sysm), oracle_ham(sysm)
    b = gh.basis(k, sysm.ecut)
    c = S.random_states(b.npw, sysm.nst, 3, S.sphere_volume_element(sysm)).astype(dtype)
    out = gh(b, DeviceArray.from_numpy(ctx, c)).numpy()
    assert rel_err(out, oh.apply_sphere(c.astype(np.complex128), b.gindex(), k)) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("natoms,nlm", [(0, 4), (1, 1), (3, 9), (20, 4)])
def test_projectors(ctx, dtype, natoms, nlm):
    """none, one channel, three groups per projector, more atoms than waves"""
    say("case: small cube projectors", natoms, nlm, np.dtype(dtype).name)
    sysm = _system((20, 18, 16), natoms, seed=1)
    v = S.local_potential(sysm)
    gh, oh = KSHamiltonian(ctx, sysm.lattice, sysm.n), orc.Ham(sysm.lattice, sysm.n)
    gh.set_scalar_potential(v)
    oh.set_potential(v)
    rng = np.random.default_rng(natoms)
    for p in sysm.positions:
        D = rng.uniform(-1, 1, (nlm, nlm))
        D = D + D.T
        gh.add_projector(p, 1.5, nlm, D, width=0.7)
        oh.add_projector_gauss(p, 1.5, nlm, 0.7, D)
    k = (0.3, 0.1, -0.2)
    b = gh.basis(k, sysm.ecut)
    c = S.random_states(b.npw, sysm.nst, 3, S.sphere_volume_element(sysm)).astype(dtype)
    out = gh(b, DeviceArray.from_numpy(ctx, c)).numpy()
    assert rel_err(out, oh.apply_sphere(c.astype(np.complex128), b.gindex(), k)) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
def test_batch_equals_single_blocks(ctx, dtype):
    """uneven blocks in one launch give the single applications bit for bit"""
    sysm = _system((16, 20, 16), 3, seed=2)
    gh = gpu_ham(ctx, sysm)
    bases, ins, outs = [], [], []
    for i, (nst, e) in enumerate([(1, 18.0), (5, 12.0), (3, 16.0)]):
        b = gh.basis((0.1 * i, 0.0, -0.2 * i), e)
        c = S.random_states(b.npw, nst, i, S.sphere_volume_element(sysm)).astype(dtype)
        bases.append(b)
        ins.append(DeviceArray.from_numpy(ctx, c))
        outs.append(DeviceArray(ctx, c.shape, dtype))
    gh.apply_batch(bases, ins, outs)
    for b, i, o in zip(bases, ins, outs):
        assert np.array_equal(o.numpy(), gh(b, i).numpy())


@pytest.mark.parametrize("dtype", DTYPES)
def test_taylor_exponential(ctx, dtype):
    """the accumulators: exp(f H) phi against the oracle's applications"""
    sysm = _system((18, 18, 18), 2, seed=3)
    gh, oh = gpu_ham(ctx, sysm), oracle_ham(sysm)
    b = gh.basis((0.0, 0.1, 0.0), sysm.ecut)
    c = S.random_states(b.npw, sysm.nst, 3, S.sphere_volume_element(sysm)).astype(dtype)
    f = -0.02j
    d = DeviceArray.from_numpy(ctx, c)
    full = rt.exponential_2_for_1(gh, b, d, f, 2 * f)
    term = c.astype(np.complex128)
    one, two = term.copy(), term.copy()
    for it in range(1, 5):
        term = oh.apply_sphere(term, b.gindex(), (0.0, 0.1, 0.0)) / it
        one, two = one + f ** it * term, two + (2 * f) ** it * term
    assert rel_err(full.numpy(), one) < TOL[dtype]
    assert rel_err(d.numpy(), two) < TOL[dtype]
