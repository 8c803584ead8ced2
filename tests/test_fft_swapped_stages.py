"""Host emulation of the swapped cross-lane stages of the split line transforms
(inq_amd/csrc/fft_reg.hpp: fft_split and fft_quad with an even number of values
per lane).  The lane exchanges are restated as what v_permlane32_swap and
v_permlane16_swap do to two registers (the upper part's value of the first and
the lower part's value of the second trade places), and the transforms run
register by register as the kernels do, so a wrong register pairing, quarter
turn, part factor or output order fails here, before any GPU run.  Also the
x passes' split of a line's point mask over a lane pair.
"""
import numpy as np
import pytest

SIZES = [12, 16, 18, 20, 24, 28, 30, 32, 36, 40, 48, 54, 60, 64, 72, 80, 96, 100, 108, 120, 128]
PAIR = [n for n in SIZES if n % 4 == 0]
QUAD = [n for n in SIZES if n % 8 == 0]


def dft(y, sign):
    n = np.arange(len(y))
    return np.exp(sign * 2j * np.pi * np.outer(n, n) / len(y)) @ y


def swap(a, b, parts):
    """a, b: one value per part; parts: (lower, upper) part indices that trade"""
    a, b = a.copy(), b.copy()
    for lo, up in parts:
        a[up], b[lo] = b[lo], a[up]
    return a, b


S32 = {2: [(0, 1)], 4: [(0, 2), (1, 3)]}
S16 = [(0, 1), (2, 3)]


def out_j(n, s, j):
    m = n // s
    return j - m // 2 + n // 2 if j >= m // 2 else j


def out_q(n, s, q):
    m = n // s
    return q * (m // 2) if s == 2 else (q >> 1) * (m // 2) + (q & 1) * m


def order(n, s):
    """[part][register] -> index of the line after dit, before dif"""
    return np.array([[out_j(n, s, j) + out_q(n, s, q) for j in range(n // s)] for q in range(s)])


def turn(t, up, sign):
    return np.where(up, 1j * sign * t, t)


def w(n, k, sign):
    return np.exp(sign * 2j * np.pi * k / n)


def part_turn(sign):
    q = np.arange(4)
    return np.where(q >= 2, w(8, 1, sign), 1.0) * np.where(q & 1, 1j * sign, 1.0)


def stage(v, n, k, up, parts, sign, rho=1.0):
    """one dit butterfly of registers k, k + M/2 (twiddle length n)"""
    half = v.shape[1] // 2
    e, o = swap(v[:, k], v[:, k + half], parts)
    t = turn(o * rho * w(n, k, sign), up, sign)
    v[:, k], v[:, k + half] = e + t, e - t


def stage_dif(v, n, k, up, parts, sign, rho=1.0):
    half = v.shape[1] // 2
    s = v[:, k] + v[:, k + half]
    d = turn((v[:, k] - v[:, k + half]) * rho * w(n, k, sign), up, sign)
    v[:, k], v[:, k + half] = swap(s, d, parts)


def dit(x, s, sign):
    n = len(x)
    v = np.array([dft(x[q::s], sign) for q in range(s)])
    q = np.arange(s)
    for k in range(n // s // 2):
        stage(v, 2 * n // s, k, q >= s // 2, S32[s], sign)
    if s == 4:
        for k in range(n // s // 2):
            stage(v, n, k, np.zeros(4, bool), S16, sign, part_turn(sign))
    return v


def dif(v, s, sign):
    n = v.size
    v = v.copy()
    q = np.arange(s)
    if s == 4:
        for k in range(n // s // 2):
            stage_dif(v, n, k, np.zeros(4, bool), S16, sign, part_turn(sign))
    for k in range(n // s // 2):
        stage_dif(v, 2 * n // s, k, q >= s // 2, S32[s], sign)
    return np.array([dft(r, sign) for r in v])


def line(n):
    rng = np.random.default_rng(n)
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


def reference(x, sign):
    return np.fft.fft(x) if sign < 0 else np.fft.ifft(x) * len(x)


CASES = [(n, 2) for n in PAIR] + [(n, 4) for n in QUAD]


@pytest.mark.parametrize("n,s", CASES)
def test_output_order_covers_the_line(n, s):
    assert sorted(order(n, s).ravel()) == list(range(n))


@pytest.mark.parametrize("n,s", CASES)
@pytest.mark.parametrize("sign", [-1, 1])
def test_dit(n, s, sign):
    x = line(n)
    assert np.allclose(dit(x, s, sign), reference(x, sign)[order(n, s)])


@pytest.mark.parametrize("n,s", CASES)
@pytest.mark.parametrize("sign", [-1, 1])
def test_dif(n, s, sign):
    x = line(n)
    ref = reference(x, sign)
    assert np.allclose(dif(x[order(n, s)], s, sign), np.array([ref[q::s] for q in range(s)]))


def test_a_wrong_part_factor_fails():
    x = line(72)
    v = np.array([dft(x[q::4], -1) for q in range(4)])
    for k in range(9):
        stage(v, 36, k, np.arange(4) >= 2, S32[4], -1)
    for k in range(9):
        stage(v, 72, k, np.zeros(4, bool), S16, -1, part_turn(1))  # the other sign's factors
    assert not np.allclose(v, reference(x, -1)[order(72, 4)])


@pytest.mark.parametrize("n", SIZES)
def test_point_mask_runs(n):
    """the runs of a line's point mask and the counts before them: the compact
    index of every point equals its rank along the line"""
    rng = np.random.default_rng(n)
    bits = rng.integers(0, 2, n)
    words = [int(sum(int(b) << i for i, b in enumerate(bits[32 * k:32 * k + 32]))) for k in range(4 if n > 96 else 3)]
    base = 7
    rank = base + np.concatenate([[0], np.cumsum(bits)[:-1]])
    runs = 2 if n % 4 == 0 else 1
    L = n // 2 // runs
    keep = (1 << L) - 1
    c = base
    for e in range(runs):
        run = []
        for h in range(2):
            b = (2 * e + h) * L
            k, o = b >> 5, b & 31
            x = words[k] >> o
            if o + L > 32 and k + 1 < len(words):
                x |= (words[k + 1] << ((32 - o) & 31)) & 0xffffffff
            run.append(x & keep)
        for h in range(2):
            cnt = c + (bin(run[0]).count("1") if h else 0)
            for k in range(L):
                j = e * L + k
                i0 = out_j(n, 2, j) + out_q(n, 2, h) if runs == 2 else j + h * (n // 2)
                bit = (run[h] >> k) & 1
                assert bit == bits[i0]
                if bit:
                    assert cnt == rank[i0]
                cnt += bit
        c += bin(run[0]).count("1") + bin(run[1]).count("1")
