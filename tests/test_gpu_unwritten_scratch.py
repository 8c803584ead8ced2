"""The Hermitian eigensolver on scratch memory that holds NaN: a factorisation of an
infinite matrix leaves NaN in every workspace array, and smaller matrices solved in
the same workspace afterwards give finite, orthonormal eigenvectors.

Tolerances as in test_gpu_eigh.py: 1e-11 for residuals and orthonormality."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import operations as ops
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 17, 20])
def test_diagonalize_after_nan(n):
    say("case: diagonalize on NaN scratch", n)
    ctx = Context(0)
    ops.diagonalize(ctx, DeviceArray.from_numpy(ctx, np.full((24, 24), np.inf, dtype=np.complex128)))
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    a = 0.5 * (a + a.conj().T)
    d = DeviceArray.from_numpy(ctx, a)
    w = ops.diagonalize(ctx, d)
    u = d.numpy().conj().T
    assert np.all(np.isfinite(u)) and np.all(np.isfinite(w))
    assert np.max(np.abs(a @ u - u * w)) < 1e-11 * max(1.0, np.max(np.abs(w)))
    assert np.max(np.abs(u.conj().T @ u - np.eye(n))) < 1e-11
