"""H on grids whose cube fits the LDS with a projector sphere that holds grid points
twice, through periodic images (its radius is above half of a box edge): alone, beside an
ordinary projector and as the second of two, s + p and d channels, against the FP64
oracle.  The one-launch kernel adds a projector's values to its points without
synchronisation, so such a projector has to take the plane and x passes; repeated
applications give the same bits.

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
@pytest.mark.parametrize("n", [(12, 12, 12), (16, 16, 12)])
@pytest.mark.parametrize("radii,nlm", [((2.0,), 4), ((2.0, 1.2), 4), ((1.2, 2.0), 4), ((2.0, 1.2), 9)])
def test_sphere_above_half_the_box(ctx, dtype, n, radii, nlm):
    say("case: repeated points", n, radii, nlm, np.dtype(dtype).name)
    L = np.diag([0.28 * x for x in n])  # 3.36 bohr along the shortest edge
    rng = np.random.default_rng(sum(n) + nlm)
    pos = rng.uniform(-0.5, 0.5, (len(radii), 3)) @ L
    gh, oh = KSHamiltonian(ctx, L, n), orc.Ham(L, n)
    v = rng.standard_normal(n[0] * n[1] * n[2])
    gh.set_scalar_potential(v)
    oh.set_potential(v)
    for p, r in zip(pos, radii):
        D = rng.uniform(-1, 1, (nlm, nlm))
        D = D + D.T
        gh.add_projector(p, r, nlm, D, width=0.7)
        oh.add_projector_gauss(p, r, nlm, 0.7, D)
    points = gh.projector_points(radii.index(2.0))[0]
    assert len(np.unique(points, axis=0)) < len(points)
    k = (0.3, 0.1, -0.2)
    b = gh.basis(k, 14.0)
    c = S.random_states(b.npw, 4, 3, np.linalg.det(L) / float(np.prod(n)) ** 2).astype(dtype)
    d = DeviceArray.from_numpy(ctx, c)
    out = gh(b, d).numpy()
    assert rel_err(out, oh.apply_sphere(c.astype(np.complex128), b.gindex(), k)) < TOL[dtype]
    assert all(np.array_equal(gh(b, d).numpy(), out) for _ in range(3))
