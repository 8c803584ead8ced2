"""Launch shapes chosen by the size of the work (states per x-pass work-group, planes
per plane-pass work-group) give the same bits as shapes set by the caller: few states
on a grid whose passes leave CUs idle, one state, d channels whose tables fill the LDS
with enough states for eight per work-group, uneven blocks, and against the oracle
the projections of a projector with three groups and of spheres with more slots than
16 lanes take in one round.

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
@pytest.mark.parametrize("n,nst,natoms,nlm,radius", [((32, 32, 32), 16, 3, 4, 1.6), ((36, 32, 32), 1, 2, 1, 1.0),
                                                     ((40, 48, 36), 17, 5, 9, 2.4), ((36, 36, 36), 40, 2, 9, 3.0)])
def test_shapes(ctx, dtype, n, nst, natoms, nlm, radius):
    say("case: launch shapes", n, nst, natoms, nlm, np.dtype(dtype).name)
    L = np.diag([0.28 * x for x in n])
    rng = np.random.default_rng(sum(n) + nst)
    pos = rng.uniform(-0.5, 0.5, (natoms, 3)) @ L
    sysm = S.System("shapes", 500 + sum(n), L, n, pos, 14.0, nst, v_sigma=0.6, kb_width=0.7, kb_radius=radius)
    gh, oh = KSHamiltonian(ctx, L, n), orc.Ham(L, n)
    v = S.local_potential(sysm)
    gh.set_scalar_potential(v)
    oh.set_potential(v)
    for p in pos:
        D = rng.uniform(-1, 1, (nlm, nlm))
        D = D + D.T
        gh.add_projector(p, radius, nlm, D, width=0.7)
        oh.add_projector_gauss(p, radius, nlm, 0.7, D)
    b = gh.basis((0.2, -0.1, 0.3), 14.0)
    phi = S.random_states(b.npw, nst, 3, S.sphere_volume_element(sysm)).astype(dtype)
    d = DeviceArray.from_numpy(ctx, phi)
    auto = gh(b, d).numpy()
    assert rel_err(auto, oh.apply_sphere(phi.astype(np.complex128), b.gindex(), (0.2, -0.1, 0.3))) < TOL[dtype]
    for xw, pb in ((1, 1), (2, 2), (4, 0), (4, 100), (8, 1)):
        gh.set_launch_shape(dtype, xw)
        gh.set_plane_batch(dtype, pb)
        assert np.array_equal(gh(b, d).numpy(), auto), (xw, pb)
