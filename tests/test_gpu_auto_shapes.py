"""Automatic launch shapes on both sides of each line of their rule give the bits of
four states per work-group: blocks whose groups of two fill the CUs or pass them, few
states in each precision, long complex128 lines, d channels whose tables leave room
for one group of four or eight, enough states for one, two and three rounds of eight,
and a batch of uneven blocks."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, KSHamiltonian
from inq_amd import systems as S
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nlm,radius,counts", [((36, 36, 36), 4, 1.8, (1, 5, 12, 13)), ((36, 32, 32), 9, 2.2, (8, 20, 33)),
                                                 ((72, 48, 40), 4, 1.6, (3, 9)), ((32, 32, 32), 9, 2.4, (64, 96, 97)),
                                                 ((40, 36, 36), 9, 2.0, (65,))])
def test_auto_equals_four(ctx, dtype, n, nlm, radius, counts):
    say("case: automatic shapes", n, nlm, counts, np.dtype(dtype).name)
    L = np.diag([0.28 * x for x in n])
    rng = np.random.default_rng(sum(n))
    gh = KSHamiltonian(ctx, L, n)
    gh.set_scalar_potential(rng.standard_normal(n[0] * n[1] * n[2]))
    for p in rng.uniform(-0.5, 0.5, (5, 3)) @ L:
        gh.add_projector(p, radius, nlm, np.diag(rng.uniform(-1, 1, nlm)), width=0.7)
    b = gh.basis((0.2, -0.1, 0.3), 14.0)
    vol = np.linalg.det(L) / (n[0] * n[1] * n[2]) ** 2
    ins = [DeviceArray.from_numpy(ctx, S.random_states(b.npw, m, m, vol).astype(dtype)) for m in counts]
    batch = [gh.basis((0.2 + 0.1 * i, 0.0, 0.0), 14.0 - i) for i in range(3)]
    bins = [DeviceArray.from_numpy(ctx, S.random_states(x.npw, 2 + 3 * i, i, vol).astype(dtype)) for i, x in enumerate(batch)]

    def run():
        outs = [DeviceArray(ctx, d.shape, dtype) for d in bins]
        gh.apply_batch(batch, bins, outs)
        return [gh(b, d).numpy() for d in ins] + [o.numpy() for o in outs]

    auto = run()
    gh.set_launch_shape(dtype, 4)
    gh.set_plane_batch(dtype, 1)
    assert all(np.array_equal(x, y) for x, y in zip(run(), auto))
