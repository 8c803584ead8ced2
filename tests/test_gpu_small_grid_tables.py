"""The tables that H reads on a grid whose cube fits the LDS belong to H: a basis that
has run the transforms alone holds none, and the first H on it allocates them (the
offset of every sphere point, four bytes each), or prepare() before it does.

200 bases of the whole 24^3 cube, without projectors: the offsets are 55 KB a basis,
the descriptor of a launch, which every first H allocates too, is below 1 KB."""
import gc

import numpy as np
import pytest
import torch

from inq_amd import Context, DeviceArray
from inq_amd import systems as S
from tests.helpers import gpu_ham, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prepared", [False, True])
def test_offsets_come_with_the_first_h(prepared):
    say("case: cube tables on first use", prepared)
    ctx = Context(0)
    sysm = S.small_config(seed=3, n=(24, 24, 24), natoms=0, nst=1, ecut=6.0)
    gh = gpu_ham(ctx, sysm)
    bases = [gh.basis((0.0, 0.0, 0.0), 1e6) for _ in range(200)]
    N = 24 ** 3
    assert bases[0].npw == N
    a, o = (DeviceArray.from_numpy(ctx, np.ones((1, N), np.complex64)) for _ in range(2))
    rs = DeviceArray(ctx, (1, N), np.complex64)
    gc.collect()
    for b in bases:
        gh.to_real(b, a, 0, rs)
        if prepared:
            gh.prepare(b, 1, np.complex64)
    ctx.sync()
    free = torch.cuda.mem_get_info()[0]
    for b in bases:
        gh.apply(b, a, o)
    ctx.sync()
    grown = free - torch.cuda.mem_get_info()[0]
    assert (grown < len(bases) * 4 * N) if prepared else (grown >= len(bases) * 4 * N)
