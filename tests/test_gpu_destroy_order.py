"""A context destroyed before its Hamiltonian, basis and captured propagator (the order in
which a garbage collector may take them): the pinned objects refuse with a status, which
they note in the context, and go once the propagator has."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import _lib
from inq_amd import real_time as rt
from inq_amd import systems as S
from tests.helpers import gpu_ham, say

pytestmark = pytest.mark.gpu


def test_context_first():
    say("case: context destroyed first")
    ctx = Context(0)
    sysm = S.small_config(seed=5, n=(20, 20, 20), natoms=2, nst=3, ecut=6.0)
    gh = gpu_ham(ctx, sysm)
    b = gh.basis((0.0, 0.0, 0.0), sysm.ecut)
    c = S.random_states(b.npw, sysm.nst, 5, S.sphere_volume_element(sysm)).astype(np.complex64)
    d = DeviceArray.from_numpy(ctx, c)
    prop = rt.Propagator(gh, [b], [d], [np.full(sysm.nst, 2.0)], dt=0.05)
    prop.step(2, graph=True)
    ctx.sync()
    d.free()
    ctx.close()
    L = _lib.lib()
    for _ in range(2):
        assert L.inqx_ham_destroy(gh.h) == _lib.INQX_ERR_STATE
        assert L.inqx_basis_destroy(b.h) == _lib.INQX_ERR_STATE
    prop.close()
    assert L.inqx_basis_destroy(b.h) == 0
    assert L.inqx_ham_destroy(gh.h) == 0
    b.h.value = gh.h.value = None
