"""The oracle's non-local operator with a projector sphere that holds grid points twice,
through periodic images: equal to a numpy sum over the sphere's points, and to itself
when repeated (several threads take part)."""
import numpy as np
import pytest

from oracle import oracle as orc


@pytest.mark.parametrize("nst", [1, 2, 5])
def test_points_twice(nst):
    n, nlm, k = (12, 12, 12), 4, (0.3, 0.1, -0.2)
    L = np.diag([0.28 * x for x in n])
    rng = np.random.default_rng(nst)
    oh = orc.Ham(L, n)
    oh.set_potential(np.zeros(int(np.prod(n))))
    D = rng.uniform(-1, 1, (nlm, nlm))
    D = D + D.T
    oh.add_projector_gauss(rng.uniform(-0.5, 0.5, 3) @ L, 2.3, nlm, 0.7, D)
    coords, _, rel, mat = oh.projector_points(0, nlm)
    assert len(np.unique(coords, axis=0)) < len(coords)
    N = int(np.prod(n))
    phi = rng.standard_normal((N, nst)) + 1j * rng.standard_normal((N, nst))
    at = (coords[:, 0] * n[1] + coords[:, 1]) * n[2] + coords[:, 2]
    ph = np.exp(1j * (rel.astype(float) @ np.array(k)))
    P = np.linalg.det(L) / N * (mat @ (ph[:, None] * phi[at]))
    want = np.zeros_like(phi)
    np.add.at(want, at, np.conj(ph)[:, None] * (mat.T @ (D @ P)))
    got = oh.apply_rs(phi, k).reshape(N, nst)
    # the kinetic term, from an operator without projectors
    bare = orc.Ham(L, n)
    bare.set_potential(np.zeros(N))
    kin = bare.apply_rs(phi, k).reshape(N, nst)
    assert np.max(np.abs(got - kin - want)) < 1e-11 * np.max(np.abs(kin))
    assert all(np.array_equal(oh.apply_rs(phi, k).reshape(N, nst), got) for _ in range(20))
