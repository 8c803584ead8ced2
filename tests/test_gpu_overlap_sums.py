"""Complex64 overlaps add at most as many products in FP32 as fit 24 bits here: the
real and imaginary parts are multiples of 1/128 in [1, 2), their products multiples
of 2^-14 below 4, so the sums of 128 complex values (256 products, below 2^10) are
exact in FP32 in any order and those of many more are not.  On blocks whose FP32 sums
end at 128 values the overlaps therefore equal the integer sums exactly: one and
several tiles, a block with itself (Hermitian) and with another one, sizes with a
remainder in every direction."""
import numpy as np
import pytest

from inq_amd import Context, DeviceArray
from inq_amd import operations as ops
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,npw", [(128, 20000), (128, 30001), (64, 120000), (65, 7003), (5, 40000)])
def test_fp32_sums_end_at_128_values(n, npw):
    say("case: overlap sums", n, npw)
    ctx = Context(0)
    rng = np.random.default_rng(n + npw)
    q = rng.integers(128, 256, (2, 2, n, npw))
    a, b = (((re + 1j * im) / 128.0).astype(np.complex64) for re, im in q)
    da, db = DeviceArray.from_numpy(ctx, a), DeviceArray.from_numpy(ctx, b)
    for x, y, u, v in ((da, da, q[0], q[0]), (da, db, q[0], q[1])):
        got = ops.overlap(ctx, x, y, 1.0).numpy()
        # products below 2^16 and sums below 2^35: exact in FP64
        p = [[(u[i].astype(float) @ v[j].astype(float).T) for j in range(2)] for i in range(2)]
        want = (p[0][0] + p[1][1] + 1j * (p[0][1] - p[1][0])) / 2.0 ** 14
        assert np.array_equal(got, want)
