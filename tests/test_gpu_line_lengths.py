"""GPU parity of the line transforms at every built length: an odd and an even
number of values per lane, over lane pairs and over four lanes, through H with
projectors (both transform orders, the point masks of both lane layouts), the
sphere -> real transforms and the plain Poisson solves.

Tolerances as in test_gpu_hamiltonian.py and test_gpu_exchange.py: 1e-11 in
complex128, 2e-5 in complex64 (max error over max reference)."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import systems as S
from tests.helpers import gpu_ham, oracle_ham, rel_err, say

pytestmark = pytest.mark.gpu

TOL = {np.complex128: 1e-11, np.complex64: 2e-5}


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


def _system(n):
    rng = np.random.default_rng(n)
    L = np.eye(3) * (0.27 * n)
    return S.System(f"len{n}", 300 + n, L, (n, n, n), rng.uniform(-0.5, 0.5, (2, 3)) @ L, 20.0, 3,
                    v_sigma=0.6, kb_width=0.7, kb_radius=1.5)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [12, 16, 18, 20, 24, 28, 30, 36, 40, 48, 54, 60])
def test_h_at_every_length(ctx, dtype, n):
    sysm = _system(n)
    k = (0.2, -0.3, 0.1)
    say("case: length", n, np.dtype(dtype).name)
    gh, oh = gpu_ham(ctx, sysm), oracle_ham(sysm)
    b = gh.basis(k, sysm.ecut)
    c = S.random_states(b.npw, sysm.nst, 3, S.sphere_volume_element(sysm)).astype(dtype)
    d = DeviceArray.from_numpy(ctx, c)
    out = gh(b, d).numpy()
    ref = oh.apply_sphere(c.astype(np.complex128), b.gindex(), k)
    assert rel_err(out, ref) < TOL[dtype]
    cube = np.zeros((sysm.nst, n ** 3), np.complex128)
    cube[:, b.gindex()] = c
    real = np.fft.ifftn(cube.reshape(-1, n, n, n), axes=(1, 2, 3)).reshape(sysm.nst, -1)
    rs = gh.to_real(b, d)
    assert rel_err(rs.numpy(), real) < TOL[dtype]
    assert rel_err(gh.to_sphere(b, rs, sysm.nst).numpy(), c) < TOL[dtype]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [18, 20, 28, 36, 54, 72, 80, 96])
def test_poisson_at_every_kind_of_length(ctx, dtype, n):
    say("case: poisson length", n, np.dtype(dtype).name)
    sysm = _system(n)
    gh = gpu_ham(ctx, sysm)
    rng = np.random.default_rng(n)
    rho = (rng.standard_normal((2, n ** 3)) + 1j * rng.standard_normal((2, n ** 3))).astype(dtype)
    out = gh.poisson(DeviceArray.from_numpy(ctx, rho)).numpy()
    m = np.fft.fftfreq(n, 1.0 / n) * 2.0 * np.pi / sysm.lattice[0, 0]
    g2 = m[:, None, None] ** 2 + m[None, :, None] ** 2 + m[None, None, :] ** 2
    kern = np.where(g2 < 1e-6, 0.0, 4.0 * np.pi / np.where(g2 < 1e-6, 1.0, g2))
    f = np.fft.fftn(rho.astype(np.complex128).reshape(-1, n, n, n), axes=(1, 2, 3)) * kern
    assert rel_err(out, np.fft.ifftn(f, axes=(1, 2, 3)).reshape(2, -1)) < TOL[dtype]
