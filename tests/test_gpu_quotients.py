"""recip(), quot() and sqrt_core() (fortrancfd_amd/csrc/fluid_coop.hpp) stand for 1 / d, n / d and sqrt(x) where the
kernels have tested the operands' range: the same bits as the host's correctly rounded operations, on operands
where a last bit is hardest to get: mantissas of ones and next to a power of two, quotients and roots within
2^-105 of the middle between two doubles.  The bar is equality."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "device", "_build", "libquotients.so")
RECIP, QUOT, ROOT = range(3)


def evaluate(op, a, b):
    lib = C.CDLL(LIB)
    a, b = (np.ascontiguousarray(x, np.float64) for x in np.broadcast_arrays(a, b))
    out = np.zeros_like(b)
    p = lambda x: x.ctypes.data_as(C.POINTER(C.c_double))
    assert lib.quotients_eval(C.c_int(op), C.c_int(b.size), p(a), p(b), p(out)) == 0
    return out


def divisors(rng):
    """Mantissas in [1, 2): all ones and its neighbours, next to 1, to 3/2 and to 4/3, and random ones."""
    k = np.arange(64)
    ints = np.concatenate([2 ** 53 - 1 - k, 2 ** 52 + k, 3 * 2 ** 51 + k - 32, 2 ** 54 // 3 + k - 32,
                           rng.integers(2 ** 52, 2 ** 53, 4000)])
    return ints.astype(np.float64) * 2.0 ** -52


def near_middle(rng, count):
    """(n, d): n / d differs from the middle between two doubles by j / d units of 2^-54, j small and odd."""
    out = []
    while len(out) < count:
        d = int(rng.integers(2 ** 52, 2 ** 53)) | 1
        if len(out) % 4 == 0:
            d = 2 ** 53 - 1 - 2 * int(rng.integers(0, 64))
        j = int(rng.choice([1, -1, 3, -3, 5, -5, 7, -7]))
        m = j * pow(d, -1, 2 ** 54) % 2 ** 54
        if m < 2 ** 53:
            continue
        n = (m * d - j) >> 54
        assert n * 2 ** 54 + j == m * d and n < 2 ** 53
        out.append((float(n), float(d)))
    a = np.array(out)
    return a[:, 0], a[:, 1] * 2.0 ** -52


def differ(got, want):
    bad = np.flatnonzero(got != want)
    return [(float(got[i]).hex(), float(want[i]).hex()) for i in bad[:4]], bad.size


def test_reciprocals():
    rng = np.random.default_rng(81)
    d = divisors(rng)
    d = np.concatenate([np.ldexp(d, e) for e in (-60, -3, 0, 1, 30, 59)])
    first, n = differ(evaluate(RECIP, 1.0, d), 1.0 / d)
    assert n == 0, (n, d.size, first)


def test_quotients():
    rng = np.random.default_rng(82)
    d = divisors(rng)
    n = np.concatenate([[1.0, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52, 1.5, 3.0 - 2.0 ** -51], rng.uniform(1.0, 2.0, 27)])
    N, D = (x.ravel() for x in np.meshgrid(n, d))
    h = near_middle(rng, 20000)
    N, D = np.concatenate([N, h[0]]), np.concatenate([D, h[1]])
    sign = rng.choice([-1.0, 1.0], N.size)
    for en, ed in ((0, 0), (-690, 20), (-100, -59), (59 - 53, 59), (59 - 53, -59)):
        a, b = np.ldexp(sign * N, en), np.ldexp(D, ed)
        first, bad = differ(evaluate(QUOT, a, b), a / b)
        assert bad == 0, (en, ed, bad, a.size, first)
    z = evaluate(QUOT, np.zeros(8), np.ldexp(d[:8], 3))
    assert (z == 0.0).all()


@pytest.mark.parametrize("species", range(3))
def test_mole_fractions(species):
    """y / (sw wt): the divisors' reciprocals are refined from products of 1 / sw and 1 / wt."""
    rng = np.random.default_rng(84 + species)
    wt = np.array([1.00797, 17.00737, 33.00677])
    h = near_middle(rng, 20000)
    d = divisors(rng)
    D = np.concatenate([np.repeat(d[:64], 24), h[1], d])
    N = np.concatenate([np.tile(np.concatenate([[1.0, 1.5, 1.25, 1.0 + 2.0 ** -52], rng.uniform(1.0, 2.0, 20)]), 64), h[0],
                        rng.uniform(1.0, 2.0, d.size)])
    sw = D / wt[species]
    for s in range(-2, 3):                                   # a sw whose product with wt is D, where there is one
        t = sw + s * np.spacing(sw)
        sw = np.where((sw * wt[species] != D) & (t * wt[species] == D), t, sw)
    assert (sw * wt[species] == D).sum() > 0.5 * D.size and (sw * wt[species] == 2.0 - 2.0 ** -52).any()
    y = rng.uniform(0.1, 1.0, (3, D.size))
    y[species] = N
    x = np.zeros_like(y)
    lib = C.CDLL(LIB)
    p = lambda v: v.ctypes.data_as(C.POINTER(C.c_double))
    assert lib.quotients_mole(C.c_int(D.size), p(wt), p(sw), p(y), p(x)) == 0
    want = y / (sw * wt[:, None])
    first, bad = differ(x.ravel(), want.ravel())
    assert bad == 0, (bad, x.size, first)


def test_roots():
    rng = np.random.default_rng(83)
    x = [divisors(rng), divisors(rng) * 2.0]
    hard = []
    for j in [8 * i + 1 for i in range(-40, 41)]:
        for want in (54, 55):                                # the root's square modulo 2^want is j
            r = 1
            for bits in range(3, want):                      # (Hensel: one more bit a time)
                if (r * r - j) % 2 ** (bits + 1):
                    r += 2 ** (bits - 1)
            assert (r * r - j) % 2 ** want == 0
            for m in {r % 2 ** want, -r % 2 ** want, (r + 2 ** (want - 1)) % 2 ** want, (-r + 2 ** (want - 1)) % 2 ** want}:
                m %= 2 ** 54
                if m >= 2 ** 53 and (m * m - j) % 2 ** want == 0 and (m * m - j) >> want < 2 ** 53:
                    hard.append(((m * m - j) >> want) * 2.0 ** (want - 54 - 52))
    assert len(hard) > 100
    x = np.concatenate(x + [np.array(hard)])
    for e in (-600, -2, 0, 2, 58):
        b = np.ldexp(x, e)
        first, n = differ(evaluate(ROOT, 1.0, b), np.sqrt(b))
        assert n == 0, (e, n, b.size, first)
