"""The automatic launch shapes can be set back: 0 is accepted for the x passes as it
is for the plane passes, other values than those of the search are refused."""
import numpy as np
import pytest

from inq_amd import Context, InqxError, KSHamiltonian


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_zero_is_the_automatic_shape(dtype):
    ham = KSHamiltonian(Context(-1), np.eye(3) * 6.0, (16, 16, 16))
    for xwaves in (4, 0, 8, 0):
        ham.set_launch_shape(dtype, xwaves)
        ham.set_plane_batch(dtype, xwaves)
    for xwaves in (-1, 3, 16):
        with pytest.raises(InqxError):
            ham.set_launch_shape(dtype, xwaves)
