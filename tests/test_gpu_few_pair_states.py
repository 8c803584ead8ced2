"""Exchange of a block of few states with its own states, where the sums over the
solved pairs run on one, two or four waves: every count around the limits of a wave's
share and of the wave counts, all occupied and with an unoccupied one, against the
form that solves every ordered pair; chunks of one row give the same bits.

Tolerances as in test_gpu_symmetric_pairs.py: complex128 1e-10, complex64 5e-5 of the
largest value."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, KSHamiltonian
from inq_amd.exchange import ExchangeOperator
from tests.helpers import rel_err, say

pytestmark = pytest.mark.gpu
TOL = {np.complex128: 1e-10, np.complex64: 5e-5}


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("nst", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("empty", [None, 0, 1])
def test_few_states(ctx, dtype, nst, empty):
    say("case: few pair states", nst, empty, np.dtype(dtype).name)
    n = (18, 12, 20)  # 4320 points, no multiple of 64
    gh = KSHamiltonian(ctx, np.diag([0.35 * x for x in n]), n)
    b = gh.basis((0, 0, 0), 8.0)
    rng = np.random.default_rng(nst)
    phi = (rng.standard_normal((nst, b.npw)) + 1j * rng.standard_normal((nst, b.npw))).astype(dtype)
    occ = rng.uniform(0.5, 2.0, nst)
    if empty is not None and nst > 1:
        occ[empty] = 0.0
    ex = ExchangeOperator(gh, b, exchange_coefficient=0.7, zeroterm=0.3)
    d = DeviceArray.from_numpy(ctx, phi)
    sym = ex.direct(d, d, occ).numpy()
    full = ex.direct(d, DeviceArray.from_numpy(ctx, phi.copy()), occ).numpy()
    assert rel_err(sym, full) < TOL[dtype]
    gh.set_exchange_workspace(1)  # one row a chunk
    one = ex.direct(d, d, occ).numpy()
    gh.set_exchange_workspace(0)
    assert np.array_equal(sym, one)
