"""Batched Poisson solves against numpy's transform where the plane passes change
form: lane pairs and four lanes per line (72 points), planes that cross LDS whole and
in two pieces (above 40 KB: 72 points complex64, 54 and 60 complex128), lines that do
not fill the last wave, square planes with another number of planes (the line pass
reads transposed planes), the largest planes and planes with n1 != n2; two densities
with a shift of G, solved in place.

Tolerances: complex128 1e-11, complex64 2e-5 of the largest value."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, KSHamiltonian
from tests.helpers import rel_err, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [(12, 48, 48), (54, 54, 54), (16, 60, 60), (20, 64, 64), (72, 72, 72), (12, 80, 80),
                               (96, 54, 54), (12, 100, 100), (16, 108, 108), (12, 120, 120), (18, 128, 128),
                               (12, 72, 80)])
def test_poisson(ctx, dtype, n):
    say("case: Poisson planes", n, np.dtype(dtype).name)
    L = np.array([0.3 * n[0], 0.31 * n[1], 0.29 * n[2]])
    gh = KSHamiltonian(ctx, np.diag(L), n)
    rng = np.random.default_rng(sum(n))
    rho = (rng.standard_normal((2,) + n) + 1j * rng.standard_normal((2,) + n)).astype(dtype)
    q = np.array([0.11, -0.07, 0.05])
    d = DeviceArray.from_numpy(ctx, rho.reshape(2, -1))
    gh.poisson(d, gshift=q)
    G = [2 * np.pi / L[k] * np.fft.fftfreq(n[k], 1.0 / n[k]) + q[k] for k in range(3)]
    g2 = G[0][:, None, None] ** 2 + G[1][None, :, None] ** 2 + G[2][None, None, :] ** 2
    f = np.fft.fftn(rho.astype(np.complex128), axes=(1, 2, 3))
    ref = np.fft.ifftn(4 * np.pi * f / g2, axes=(1, 2, 3)).reshape(2, -1)
    assert rel_err(d.numpy(), ref) < (1e-11 if dtype == np.complex128 else 2e-5)
