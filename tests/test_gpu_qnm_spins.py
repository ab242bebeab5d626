"""Kerr QNM roots of remnants with high spin: their error against extended precision
beside that of the same continued fractions evaluated term by term in double
precision."""
import numpy as np
import pytest

from eobgpu_amd import eobstuff as ES
from eobgpu_amd import pipeline as P

pytestmark = pytest.mark.gpu

ANG, RAD = 60, 300   # terms of the two fractions


def fraction(beta, ag):
    t = beta[-1]
    for b, g in zip(beta[-2::-1], ag[::-1]):
        t = b - g / t
    return t


def angular(A, c, m, F):
    k1, k12 = F(abs(m + 2)) / 2, F(abs(m + 2) + abs(m - 2)) / 2
    n = np.arange(ANG + 1, dtype=F)[:, None]
    beta = n * (n - 1) + 2 * n * (k12 + 1 - 2 * c) - (2 * c * (2 * k1 - 1) - k12 * (k12 + 1)) - (c * c + 2 + A)
    return fraction(beta, (-2 * (n + 1) * (n + 2 * k1 + 1))[:-1] * (2 * (n + k12 - 2) * c)[1:])


def radial(w, a, m, A, F):
    b, I, n = np.sqrt(1 - 4 * a * a), 1j, np.arange(RAD + 1, dtype=F)[:, None]
    q = 2 / b * (I * (w / 2 - a * m))
    c0, c1, c2 = 3 - I * w - q, -4 + 2 * (2 + b) * (I * w) + 2 * q, 1 - 3 * I * w - q
    f4 = (4 * w + 2 * I) * (w / 2 - a * m) / b
    c3 = w * w * (4 + 2 * b - a * a) - 2 * a * m * w + 1 + (2 + b) * I * w - A + f4
    c4 = -1 - 2 * w * w + I * w - f4
    al, be, ga = n * n + n + c0 * n + c0, -2 * n * n + 2 * n + c1 * n + c3, n * n - 3 * n + 2 + c2 * n + c4 - c2
    return fraction(be, al[:-1] * ga[1:])


def secant(f, x, dx, steps, tol):
    y = x + dx
    fx, fy, live = f(x), f(y), np.ones(x.shape, bool)
    for _ in range(steps):
        d = fy - fx
        live = live & (d != 0)
        z = np.where(live, y - fy * (y - x) / np.where(d == 0, 1, d), y)
        fz = f(z)
        x, fx, y, fy, live = (np.where(live, y, x), np.where(live, fy, fx), z, np.where(live, fz, fy),
                              live & (np.abs(z - y) > tol * (1 + np.abs(z))))
    return y


def root(l, m, a, w, F, steps):
    """Leaver's root near w (his units, 2 M = 1) at spins a"""
    eps = float(np.finfo(F).eps)

    def f(w):
        A = secant(lambda A: angular(A, a * w, m, F), np.full_like(w, l * (l + 1) - 2), w.dtype.type(1e-3 + 1e-3j), 12, 50 * eps)
        return radial(w, a, m, A, F)
    return secant(f, w, w.dtype.type(1e-6 - 1e-6j), steps, 5 * eps)


@pytest.mark.parametrize("l,m", P.REFERENCE_MODES)
@pytest.mark.parametrize("lo,hi", [(0.8, 0.97), (0.97, 0.99)])
def test_high_spin_roots_are_as_good_as_the_serial_fractions(dev, l, m, lo, hi):
    rng = np.random.default_rng(l * 10 + m)
    af = rng.uniform(lo, hi, 160) * np.where(np.arange(160) % 2, 1.0, -1.0)
    got = np.asarray(ES.compute_QNM(l, m, 0, af, np.ones(af.size)))
    with np.errstate(all="ignore"):
        w = 2 * np.conj(np.conj(got))
        want = root(l, m, (af / 2).astype(np.longdouble), w.astype(np.clongdouble), np.longdouble, 5)
        serial = root(l, m, af / 2, (want * (1 + 1e-7)).astype(np.complex128), np.float64, 8)

    def rms(x):
        return float(np.sqrt(np.mean((np.abs(x - want) / np.abs(want)) ** 2)))
    # 160 spins: the two rms, of the same roundings met in another order, scatter by about 1 / sqrt(160)
    assert rms(w) <= 1.25 * rms(serial)
