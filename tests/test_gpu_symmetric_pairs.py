"""Exchange of a block with its own states (each unordered pair of occupied states
solved once, both states' sums taken from one read of it) against the form that
solves every ordered pair: one state, blocks that end inside and at the end of a
wave's share and of a pass over the rows (8, 16, 32, 64 and 128 states), more than
one pass, unoccupied states among them, no occupied state but one, a point count
that is no multiple of 64, planes with n1 != n2, and chunks of one row, which must
give the same bits.

Tolerances as for the other exchange sums: complex128 1e-10, complex64 5e-5 of the
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
@pytest.mark.parametrize("n,nst", [((12, 12, 12), 1), ((18, 12, 12), 8), ((18, 12, 12), 9), ((12, 12, 12), 17),
                                   ((18, 18, 18), 33), ((12, 12, 16), 65), ((18, 12, 12), 129), ((12, 12, 12), 261)])
@pytest.mark.parametrize("occupied", ["all", "some", "one"])
def test_symmetric_equals_full(ctx, dtype, n, nst, occupied):
    say("case: symmetric pairs", n, nst, occupied, np.dtype(dtype).name)
    gh = KSHamiltonian(ctx, np.diag([0.35 * x for x in n]), n)
    b = gh.basis((0, 0, 0), 8.0)
    rng = np.random.default_rng(nst)
    phi = (rng.standard_normal((nst, b.npw)) + 1j * rng.standard_normal((nst, b.npw))).astype(dtype)
    occ = rng.uniform(0.5, 2.0, nst)
    if occupied == "some":
        occ[1:][rng.uniform(size=nst - 1) < 0.4] = 0.0
    elif occupied == "one":
        occ[np.arange(nst) != nst // 2] = 0.0
    ex = ExchangeOperator(gh, b, exchange_coefficient=0.7, zeroterm=0.3)
    d = DeviceArray.from_numpy(ctx, phi)
    sym = ex.direct(d, d, occ).numpy()
    full = ex.direct(d, DeviceArray.from_numpy(ctx, phi.copy()), occ).numpy()
    assert rel_err(sym, full) < TOL[dtype]
    gh.set_exchange_workspace(1)  # one row a chunk
    one = ex.direct(d, d, occ).numpy()
    gh.set_exchange_workspace(0)
    assert np.array_equal(sym, one)
