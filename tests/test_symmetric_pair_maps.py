"""Host emulation of two index maps of the pair kernels (inq_amd/csrc/exx_kernels.hip):
k_pair_reduce_both's shares of the states (bits act and conj of a wave's states for a
row) take every solved pair's two terms exactly once, and pair_product_item gives
every (row, plane, state) to one work-group."""
import itertools

import numpy as np
import pytest

W = 8


@pytest.mark.parametrize("U", [2, 4, 8, 16])
@pytest.mark.parametrize("nst", [1, 7, 8, 9, 16, 17, 33, 64, 65, 128, 129, 300])
def test_terms_of_every_row(U, nst):
    rng = np.random.default_rng(nst * U)
    for occ in (np.ones(nst, int), (rng.uniform(size=nst) < 0.6).astype(int)):
        rows = [j for j in range(nst) if occ[j]]
        for j in rows[:3] + rows[len(rows) // 2 : len(rows) // 2 + 3] + rows[-3:]:
            w_terms, wb_terms = [], []
            for base, wave in itertools.product(range(0, nst, W * U), range(W)):
                valid = sum(1 << u for u in range(U) if base + u * W + wave < nst)
                om = sum(1 << u for u in range(U) if base + u * W + wave < nst and occ[base + u * W + wave])
                le = j - base - wave

                def mask(x):  # bits of the states with index difference <= x
                    if x < 0:
                        return 0
                    return 0xFFFFFFFF if x // W >= U - 1 else (2 << (x // W)) - 1

                act, conj = valid & (~om | mask(le)), om & mask(le - 1)
                w_terms += [base + u * W + wave for u in range(U) if (act >> u) & 1]
                wb_terms += [base + u * W + wave for u in range(U) if (conj >> u) & 1]
                assert conj & ~act == 0  # a conjugate term's pair is read
                if j <= base:
                    assert conj == 0  # rows whose sum is not added hold no term
            assert sorted(w_terms) == [i for i in range(nst) if not (occ[i] and i > j)]
            assert sorted(wb_terms) == [s for s in range(j) if occ[s]]


def test_product_items_cover_every_plane_once():
    nst, nj, n0 = 5, 3, 7
    wg = np.arange(nst * nj * n0)
    items = set(zip((wg // nst) % nj, (wg // nst) // nj, wg % nst))
    assert items == set(itertools.product(range(nj), range(n0), range(nst)))
