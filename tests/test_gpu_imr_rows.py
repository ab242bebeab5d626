"""The merger-ringdown template as a sum over its modes (more modes than one build
of its kernel holds, modes given twice and in any order, series cut inside the
inspiral and the ringdown), and the Kerr QNM roots against one secant solve in
extended precision."""
import numpy as np
import pytest
import torch

from eobgpu_amd import configs
from eobgpu_amd import eobstuff as ES
from eobgpu_amd import pipeline as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def batch(dev):
    p = configs.small_batch(n=3, seed=31)
    b = P.EOBBatch(P.make_additional_args(p["m1"], p["m2"], p["chi1"], p["chi2"]), max_step=4096, device=dev)
    b.initial_conditions(np.full(3, 10.5))
    b.integrate(rtol=1e-10, atol=1e-10, two_pass=True)
    return b, p["m1"] + p["m2"]


def template(batch, modes, N, dt=1.0 / 16384):
    b, M = batch
    b.hlm_modes_knots(modes)
    b.build_mode_splines()
    hp, hc = b.imr_template(M, dt, N)
    return (hp + 1j * hc).cpu().numpy(), b.nsamp.cpu().numpy(), b.imr["bini"].cpu().numpy()


@pytest.mark.parametrize("modes", [((5, 5), (2, 1), (2, 2), (4, 4), (3, 3)),
                                   ((3, 3), (2, 2), (5, 5), (2, 2), (2, 1), (4, 4), (3, 3), (2, 1))])
def test_template_is_the_sum_of_its_modes(batch, modes):
    n0 = 1 << 14
    _, _, bini = template(batch, ((2, 2),), n0)
    idx, nadd = int(bini[0, 1]), int(bini[0, 2])
    for N in (n0 + 1, idx + 1, idx, idx + nadd // 2, 333):
        one = {lm: template(batch, (lm,), N) for lm in set(modes)}
        h, ns, _ = template(batch, modes, N)
        want = sum(one[lm][0] for lm in modes)
        scale = sum(np.abs(one[lm][0]).max() for lm in modes)
        # each mode is a few dozen operations on phases below 2^12 (an ulp 9e-13, times m)
        assert np.abs(h - want).max() < 1e-11 * scale
        np.testing.assert_array_equal(ns, one[(2, 2)][1])


def refined_root(l, m, a, w):
    """One secant solve of Leaver's fractions from w (his units, 2 M = 1) in extended precision."""
    C, F = np.clongdouble, np.longdouble
    s, a = -2, F(a)
    k1, k12 = F(abs(m - s)) / 2, F(abs(m - s) + abs(m + s)) / 2

    def fraction(beta, alpha, gamma, depth):
        t = beta(F(depth))
        for n in range(depth - 1, -1, -1):
            t = beta(F(n)) - alpha(F(n)) * gamma(F(n + 1)) / t
        return t

    def angular(A, c):
        return fraction(lambda n: n * (n - 1) + 2 * n * (k12 + 1 - 2 * c) - (2 * c * (2 * k1 + s + 1) - k12 * (k12 + 1)) - (c * c + s * (s + 1) + A),
                        lambda n: -2 * (n + 1) * (n + 2 * k1 + 1), lambda n: 2 * (n + k12 + s) * c, 60)

    def secant(f, x, y, steps):
        fx, fy = f(x), f(y)
        for _ in range(steps):
            if fx == fy:
                break
            x, y, fx = y, y - fy * (y - x) / (fy - fx), fy
            fy = f(y)
        return y

    def radial(w):
        A = secant(lambda A: angular(A, a * w), C(l * (l + 1) - 2), C(l * (l + 1) - 2 + 1e-3 + 1e-3j), 12)
        b, I = np.sqrt(1 - 4 * a * a), C(1j)
        q = 2 * I * (w / 2 - a * m) / b
        c0, c1, c2 = 1 - s - I * w - q, -4 + 2 * I * w * (2 + b) + 2 * q, s + 3 - 3 * I * w - q
        f4 = (4 * w + 2 * I) * (w / 2 - a * m) / b
        c3 = w * w * (4 + 2 * b - a * a) - 2 * a * m * w - s - 1 + (2 + b) * I * w - A + f4
        c4 = s + 1 - 2 * w * w - (2 * s + 3) * I * w - f4
        return fraction(lambda n: -2 * n * n + (c1 + 2) * n + c3, lambda n: n * n + (c0 + 1) * n + c0, lambda n: n * n + (c2 - 3) * n + c4 - c2 + 2, 300)

    return secant(radial, C(w), C(w) * (1 + F(1e-7)), 4)


@pytest.mark.parametrize("l,m", P.REFERENCE_MODES)
def test_qnm_roots_against_extended_precision(dev, l, m):
    af = np.array([-0.97, -0.8, -0.3, 0.0, 0.2, 0.4999, 0.7, 0.85, 0.97])
    got = ES.compute_QNM(l, m, 0, af, np.ones(af.size))
    want = np.array([complex(refined_root(l, m, a / 2, 2 * g) / 2) for a, g in zip(af, got)])
    # 300 terms of the fraction, each rounded once, near |a| = 1: below 1e-14 of the root
    assert np.abs(got - want).max() < 1e-14 * np.abs(want).min()
