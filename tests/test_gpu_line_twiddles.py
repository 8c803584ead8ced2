"""Lines split over four lanes turn a value by one rounded factor.

The density of a plane wave of one step along i0, complex64, on grids whose lengths are
powers of two: every transform value before the last stage is 0 or 1, the 1/N scaling is
exact, so the density is the sum of the squares of the float32 cosine and sine of
2 pi i0 / n0, exactly, in FP64."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, KSHamiltonian
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n0", [16, 32, 64, 128])
def test_plane_wave_density(n0):
    say("case: plane wave density", n0)
    ctx = Context(0)
    n = (n0, 16, 16)
    gh = KSHamiltonian(ctx, np.diag([0.3 * x for x in n]), n)
    b = gh.basis((0.0, 0.0, 0.0), 12.0)
    c = np.zeros((1, b.npw), np.complex64)
    c[0, list(b.gindex()).index(256)] = 1.0
    N = n0 * 256
    den = gh.density_add(b, DeviceArray.from_numpy(ctx, c), np.ones(1),
                         density=DeviceArray.from_numpy(ctx, np.zeros(N))).numpy()
    arg = 2.0 * np.pi * np.arange(n0) / n0
    cos, sin = (np.float32(f(arg)).astype(np.float64) for f in (np.cos, np.sin))
    # the quarter points, where the factor is 0 or 1
    cos[n0 // 4 :: n0 // 2], sin[:: n0 // 2] = 0.0, 0.0
    assert np.array_equal(den.reshape(n0, 256), np.repeat(((cos ** 2 + sin ** 2) / N ** 2)[:, None], 256, axis=1))
