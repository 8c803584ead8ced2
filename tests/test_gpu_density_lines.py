"""Spin density of sphere states (line transform and sum over the states in one
pass) against numpy's transform in 64 bits: four lanes and two lanes per line,
planes whose lines do not fill the last wave, one state, ranges of states that do
not divide, more states than one set of occupations holds, two components, and a
sphere that fills the box.

Tolerance of the largest value of the density.  complex128: 1e-12.  complex64: the
relative error of a value of phi is at most about log2(N) butterflies' roundings,
18 x 6e-8 of the largest value, |phi|^2 twice that: 5e-6."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import systems as S
from tests.helpers import gpu_ham, rel_err, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


CASES = [((12, 12, 12), 1, 18.0), ((18, 20, 16), 7, 18.0), ((54, 12, 18), 5, 18.0), ((60, 18, 12), 5, 18.0),
         ((100, 12, 12), 3, 18.0), ((128, 16, 12), 3, 18.0), ((72, 20, 20), 37, 18.0), ((16, 16, 16), 300, 9.0),
         ((20, 12, 16), 4, 1e30), ((30, 12, 16), 4, 1e30)]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nst,ecut", CASES)
def test_density(ctx, dtype, n, nst, ecut):
    say("case: density", n, nst, ecut, np.dtype(dtype).name)
    L = np.diag([0.28 * x for x in n])
    sysm = S.System("lines", 300 + sum(n), L, n, np.zeros((0, 3)), ecut, nst, v_sigma=0.6)
    gh = gpu_ham(ctx, sysm)
    b = gh.basis((0.1, 0.0, -0.2), ecut)
    rng = np.random.default_rng(nst)
    c = (rng.standard_normal((nst, b.npw)) + 1j * rng.standard_normal((nst, b.npw))).astype(dtype)
    occ = rng.uniform(0.0, 2.0, nst)
    start = rng.uniform(0.0, 1e-3, (sysm.N, 2))
    den = DeviceArray.from_numpy(ctx, start)
    gh.density_add(b, DeviceArray.from_numpy(ctx, c), occ, den, ncomp=2, ispin=1)
    cube = np.zeros((nst, sysm.N), dtype=np.complex128)
    cube[:, b.gindex()] = c
    rs = np.fft.ifftn(cube.reshape((nst,) + n), axes=(1, 2, 3)).reshape(nst, sysm.N)
    ref = start[:, 1] + np.sum(occ[:, None] * np.abs(rs) ** 2, 0)
    got = den.numpy()
    assert np.array_equal(got[:, 0], start[:, 0])
    assert rel_err(got[:, 1], ref) < (1e-12 if dtype == np.complex128 else 5e-6)
