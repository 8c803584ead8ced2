"""H on a basis that a captured propagation graph uses: a precision or a form of H
whose tables the graph does not read still runs after the capture, as it does before
it, and the graph's next steps are those of a run without the call in between.

Cases: complex128 H beside a complex64 graph and the other way round, on a grid that
runs the plane passes and one whose cube fits the LDS, also after the vector
potential has changed before the capture (tables of both precisions of the old one).

Tolerances as in test_gpu_hamiltonian.py: 1e-11 complex128, 2e-5 complex64."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import real_time as rt
from inq_amd import systems as S
from tests.helpers import gpu_ham, oracle_ham, rel_err, say

pytestmark = pytest.mark.gpu
TOL = {np.complex128: 1e-11, np.complex64: 2e-5}
K = (0.3, -0.2, 0.45)


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("n", [(20, 20, 20), (24, 24, 24), (36, 32, 32)])
@pytest.mark.parametrize("graph_type,other", [(np.complex64, np.complex128), (np.complex128, np.complex64)])
@pytest.mark.parametrize("kick", [False, True])
def test_h_beside_a_captured_graph(ctx, n, graph_type, other, kick):
    say("case: pinned basis", n, np.dtype(graph_type).name, kick)
    sysm = S.small_config(seed=11, n=n, natoms=3, nst=4, ecut=6.0)
    gh = gpu_ham(ctx, sysm)
    b = gh.basis(K, sysm.ecut)
    c = S.random_states(b.npw, sysm.nst, 5, S.sphere_volume_element(sysm))
    for t in (graph_type, other):
        gh.prepare(b, sysm.nst, t)
    A = (0.0, 0.0, 0.0)
    if kick:
        for t in (graph_type, other):
            gh(b, DeviceArray.from_numpy(ctx, c.astype(t)))
        A = (-0.1, 0.05, 0.0)
        gh.uniform_vector_potential = np.array(A)
    phis = [DeviceArray.from_numpy(ctx, c.astype(graph_type)) for _ in range(2)]
    props = [rt.Propagator(gh, [b], [p], [np.full(sysm.nst, 2.0)], dt=0.05) for p in phis]
    ins = c.astype(other)
    try:
        props[0].step(2, graph=True)  # eager, then captured: the basis is pinned
        out = gh(b, DeviceArray.from_numpy(ctx, ins)).numpy()
        props[0].step(2, graph=True)
        props[1].step(4, graph=False)
        ends = [p.numpy() for p in phis]
    finally:
        for p in props:
            p.close()
    ref = oracle_ham(sysm).apply_sphere(ins.astype(np.complex128), b.gindex(), np.add(K, A))
    assert rel_err(out, ref) < TOL[other]
    assert np.array_equal(ends[0], ends[1])
