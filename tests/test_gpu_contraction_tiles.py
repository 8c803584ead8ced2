"""GPU parity of the overlap and rotation products at the edges of their 64 x 64
tiles and 16- or 8-value stages: the Hermitian overlap of a block with itself
(tiles on and below the diagonal), chunks of the contraction longer than one
FP32 accumulation, and the in-place triangular rotation of orthogonalize.

References: numpy in complex128.  Tolerances as in test_gpu_linalg.py: overlaps
1e-13 (complex128) and 2e-6 (complex64) of the largest value; orthogonalised
states 1e-11 and 5e-5."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import operations as ops
from tests.helpers import rel_err, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


DTYPES = [(np.complex128, 1e-13), (np.complex64, 2e-6)]


@pytest.mark.parametrize("dtype,tol", DTYPES)
@pytest.mark.parametrize("n,npw", [(1, 1), (3, 7), (64, 16), (65, 129), (130, 1000), (200, 100001)])
def test_hermitian_overlap(ctx, dtype, tol, n, npw):
    say("case: overlap of a block with itself", n, npw, np.dtype(dtype).name)
    a = _rand((n, npw), n).astype(dtype)
    d = DeviceArray.from_numpy(ctx, a)
    w = a.astype(np.complex128)
    assert rel_err(ops.overlap(ctx, d, d, 0.37).numpy(), 0.37 * (w.conj() @ w.T)) < tol


@pytest.mark.parametrize("dtype,tol", DTYPES)
@pytest.mark.parametrize("n1,n2,npw", [(1, 65, 15), (64, 64, 17), (129, 2, 4097), (70, 200, 90001)])
def test_general_overlap(ctx, dtype, tol, n1, n2, npw):
    say("case: overlap", n1, n2, npw, np.dtype(dtype).name)
    a, b = _rand((n1, npw), 1).astype(dtype), _rand((n2, npw), 2).astype(dtype)
    out = ops.overlap(ctx, DeviceArray.from_numpy(ctx, a), DeviceArray.from_numpy(ctx, b), 0.37).numpy()
    assert rel_err(out, 0.37 * (a.astype(np.complex128).conj() @ b.astype(np.complex128).T)) < tol


@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-11), (np.complex64, 5e-5)])
@pytest.mark.parametrize("n,npw", [(1, 63), (16, 64), (64, 333), (65, 641), (130, 1025)])
def test_orthogonalize(ctx, dtype, tol, n, npw):
    say("case: orthogonalize", n, npw, np.dtype(dtype).name)
    a = _rand((n, npw), n + 5).astype(dtype)
    w = a.astype(np.complex128)
    L = np.linalg.cholesky(0.013 * (w.conj() @ w.T))
    d = DeviceArray.from_numpy(ctx, a)
    ops.orthogonalize(ctx, d, 0.013)
    assert rel_err(d.numpy(), np.linalg.solve(L.conj(), w)) < tol


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_orthogonalize_leaves_a_dependent_block_alone(ctx, dtype):
    """a singular overlap is a status, and the states are as they were"""
    from inq_amd import InqxError
    a = _rand((70, 300), 4).astype(dtype)
    a[69] = 0.0
    d = DeviceArray.from_numpy(ctx, a)
    with pytest.raises(InqxError) as e:
        ops.orthogonalize(ctx, d, 1.0)
    assert "status -4" in str(e.value)
    assert np.array_equal(d.numpy(), a)


@pytest.mark.parametrize("dtype,tol", DTYPES)
@pytest.mark.parametrize("n,npw", [(1, 65), (64, 64), (129, 200)])
def test_rotations(ctx, dtype, tol, n, npw):
    say("case: rotate", n, npw, np.dtype(dtype).name)
    phi, psi, rot = _rand((n, npw), 5).astype(dtype), _rand((n, npw), 6).astype(dtype), _rand((n, n), 7)
    w = phi.astype(np.complex128)
    d = DeviceArray.from_numpy(ctx, phi)
    r = DeviceArray.from_numpy(ctx, rot)
    out = DeviceArray.from_numpy(ctx, psi)
    ops.rotate_add(ctx, r, d, out, alpha=0.5 - 1j, beta=0.25j)
    assert rel_err(out.numpy(), (0.5 - 1j) * (rot.T @ w) + 0.25j * psi.astype(np.complex128)) < 10 * tol
    ops.rotate(ctx, r, d)
    assert rel_err(d.numpy(), rot.conj() @ w) < 10 * tol
