"""Cholesky factors of matrices of two panels, which two launches leave in place, and
of one and three panels beside them: the last tile's rows around the steps it takes (8,
16 and 32), the upper triangle zero, the inverse of the factor, and the first leading
minor that is not positive definite in either panel.

Tolerance: the factor's backward error is at most about n eps |S|; 1e-12 is relative to
the largest value with n <= 65 and condition numbers below 100."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray, InqxError
from inq_amd import operations as ops
from tests.helpers import rel_err, say

pytestmark = pytest.mark.gpu


def _matrix(n):
    rng = np.random.default_rng(n)
    m = rng.standard_normal((n, 4 * n)) + 1j * rng.standard_normal((n, 4 * n))
    return m @ m.conj().T / (8 * n)


@pytest.mark.parametrize("n", [1, 5, 31, 32, 33, 39, 40, 41, 47, 48, 49, 63, 64, 65])
def test_factor_and_inverse(n):
    say("case: cholesky", n)
    ctx = Context(0)
    s = _matrix(n)
    want = np.linalg.cholesky(s)
    d = DeviceArray.from_numpy(ctx, s)
    got = ops.cholesky(ctx, d).numpy()
    assert rel_err(got, want) < 1e-12
    assert np.all(got[np.triu_indices(n, 1)] == 0)
    inv = ops.invert_triangular(ctx, d).numpy()
    assert rel_err(inv, np.linalg.inv(want)) < 1e-12
    assert np.all(inv[np.triu_indices(n, 1)] == 0)


@pytest.mark.parametrize("n,minor", [(40, 12), (40, 32), (40, 33), (50, 50), (64, 40)])
def test_first_minor(n, minor):
    say("case: cholesky minor", n, minor)
    ctx = Context(0)
    s = _matrix(n)
    s[minor - 1, minor - 1] = -1.0
    with pytest.raises(InqxError) as e:
        ops.cholesky(ctx, DeviceArray.from_numpy(ctx, s))
    assert f"minor {minor} " in str(e.value)
