"""Complex128 lines of many states: every store must write the value it was
given, whatever the wave computes next.  All states of the block are the same,
so that every row of the result equals the first bit for bit, and the first is
held against the FP64 oracle (1e-11, max error over max reference, as in
test_gpu_hamiltonian.py).  54 and 108 points: lines over a lane pair and over
four lanes whose stores are spread over the transform's last stage."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import systems as S
from tests.helpers import gpu_ham, oracle_ham, rel_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nst,passes", [(54, 52, 6), (72, 48, 4), (108, 20, 3)])
def test_equal_states_stay_equal(n, nst, passes):
    say("case: equal states", n, nst)
    ctx = Context(0)
    rng = np.random.default_rng(n)
    L = np.eye(3) * (0.29 * n)
    sysm = S.System(f"eq{n}", 300 + n, L, (n, n, n), rng.uniform(-0.5, 0.5, (4, 3)) @ L, 20.0, 1,
                    v_sigma=0.6, kb_width=0.7, kb_radius=1.5)
    k = (0.3, -0.5, 0.4)
    gh, oh = gpu_ham(ctx, sysm), oracle_ham(sysm)
    b = gh.basis(k, sysm.ecut)
    c = S.random_states(b.npw, 1, 3, S.sphere_volume_element(sysm)).astype(np.complex128)
    d = DeviceArray.from_numpy(ctx, np.repeat(c, nst, axis=0))
    ref = oh.apply_sphere(c, b.gindex(), k)
    for _ in range(passes):
        out = gh(b, d).numpy()
        assert (out == out[:1]).all(), "states %s" % np.nonzero((out != out[:1]).any(axis=1))[0]
        assert rel_err(out[:1], ref) < 1e-11
