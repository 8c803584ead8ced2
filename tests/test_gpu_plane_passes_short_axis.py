"""H through the plane and x passes on grids with a short first axis whose cube is too
large for one work-group's LDS (cubes of these lengths run in one launch instead): every
first length up to 24, square and other planes, s + p and d channels, k != 0, against the
FP64 oracle, with the same bits for every launch shape and from the autotuner's.

Tolerances as in test_gpu_hamiltonian.py: 1e-11 complex128, 2e-5 complex64."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, KSHamiltonian
from inq_amd import systems as S
from oracle import oracle as orc
from tests.helpers import rel_err, say

pytestmark = pytest.mark.gpu
TOL = {np.complex128: 1e-11, np.complex64: 2e-5}


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nlm", [((12, 48, 48), 4), ((16, 40, 48), 9), ((16, 40, 40), 4), ((18, 54, 54), 4),
                                   ((20, 48, 40), 4), ((20, 36, 40), 9), ((24, 48, 60), 4), ((24, 36, 36), 1)])
def test_h_and_shapes(ctx, dtype, n, nlm):
    say("case: short first axis", n, nlm, np.dtype(dtype).name)
    L = np.diag([0.28 * x for x in n])
    rng = np.random.default_rng(sum(n))
    pos = rng.uniform(-0.5, 0.5, (4, 3)) @ L
    nst = 5
    sysm = S.System("short", 600 + sum(n), L, n, pos, 14.0, nst, v_sigma=0.6, kb_width=0.7, kb_radius=1.6)
    gh, oh = KSHamiltonian(ctx, L, n), orc.Ham(L, n)
    v = S.local_potential(sysm)
    gh.set_scalar_potential(v)
    oh.set_potential(v)
    for p in pos:
        D = rng.uniform(-1, 1, (nlm, nlm))
        D = D + D.T
        gh.add_projector(p, 1.6, nlm, D, width=0.7)
        oh.add_projector_gauss(p, 1.6, nlm, 0.7, D)
    k = (0.2, -0.1, 0.3)
    b = gh.basis(k, 14.0)
    c = S.random_states(b.npw, nst, 3, S.sphere_volume_element(sysm)).astype(dtype)
    d = DeviceArray.from_numpy(ctx, c)
    auto = gh(b, d).numpy()
    assert rel_err(auto, oh.apply_sphere(c.astype(np.complex128), b.gindex(), k)) < TOL[dtype]
    for xw, pb in ((1, 1), (2, 3), (4, 0), (8, 2), (0, 100)):
        gh.set_launch_shape(dtype, xw)
        gh.set_plane_batch(dtype, pb)
        assert np.array_equal(gh(b, d).numpy(), auto), (xw, pb)
    (xw, pb), ms = gh.autotune_batch([b], [nst], dtype, None)
    assert xw in (1, 2, 4, 8) and pb >= 1 and ms > 0
    assert np.array_equal(gh(b, d).numpy(), auto)
