"""The tiled spline builders at the edges of their tiles, of the rows a lane owns
and of the halos, against the same not-a-knot system solved in extended precision, on even,
trajectory-like, random and graded knots ("steep": the short halo is not enough).
(scipy's own coefficients are 1.7e-10 off the extended-precision ones where
graded spacings jump back to 1, so they are no oracle for these knots.)"""
import numpy as np
import pytest
import torch

from eobgpu_amd import pipeline as P, pytdinterp
from eobgpu_amd._lib import call, lib

pytestmark = pytest.mark.gpu


def knots_of(kind, n, rng):
    if kind == "even":
        return np.arange(n) * 0.37
    if kind == "step":      # the fixed-step pass after an adaptive one
        return np.cumsum(np.where(np.arange(n) < n // 2, 33.0, 1.0))
    if kind == "random":
        return np.cumsum(rng.uniform(0.01, 1.0, n))
    if kind == "graded":
        return np.cumsum(0.8 ** (np.arange(n) % 80))
    # halving spacings damp a cut by 0.36 a row: 32 rows leave 4e-15 of it
    return np.cumsum(0.5 ** (np.arange(n) % 45))


def extended_spline(t, y):
    """(c1, c2, c3, last slope) of the not-a-knot splines of y's columns, eliminated in extended precision."""
    t, y = t.astype(np.longdouble), y.astype(np.longdouble)
    n = len(t)
    dx = np.diff(t)[:, None]
    m = np.diff(y, axis=0) / dx
    pc, pd = np.zeros((n, 1), np.longdouble), np.zeros((n, y.shape[1]), np.longdouble)
    for i in range(n):
        if i in (0, n - 1):
            j = 0 if i == 0 else n - 3
            p, q, u, v = dx[j], dx[j + 1], m[j], m[j + 1]
            e = p + q
            b, ud, dg, ld = ((((p + 2 * e) * q * u + p * p * v) / e, e, q, 0) if i == 0
                             else ((q * q * u + (2 * e + q) * p * v) / e, 0, p, e))
        else:
            b, ud, dg, ld = 3 * (dx[i] * m[i - 1] + dx[i - 1] * m[i]), dx[i - 1], 2 * (dx[i] + dx[i - 1]), dx[i]
        den = dg - (ld * pc[i - 1] if i else 0)
        pc[i], pd[i] = ud / den, (b - (ld * pd[i - 1] if i else 0)) / den
    s = pd
    for i in range(n - 2, -1, -1):
        s[i] -= pc[i] * s[i + 1]
    tt = (s[:-1] + s[1:] - 2 * m) / dx
    return s[:-1], (m - s[:-1]) / dx - tt, tt / dx, s[-1]


def exact_slopes_error(t, y, got, nser):
    """largest error of c1 dx, c2 dx^2, c3 dx^3 in units of max |y|"""
    dx = np.diff(t)
    worst = 0.0
    c = extended_spline(t, y)
    for q in range(nser):
        scale = np.abs(y[:, q]).max()
        for k in (1, 2, 3):
            worst = max(worst, float(np.max(np.abs(got[:-1, 4 * q + k] - c[k - 1][:, q]) * dx ** k) / scale))
        assert np.array_equal(got[:, 4 * q], y[:, q])
    return worst


@pytest.mark.parametrize("kind", ["even", "step", "random", "graded", "steep"])
@pytest.mark.parametrize("nser", [3])
def test_batched_builder_tile_edges(dev, kind, nser):
    lens = [4, 5, 15, 16, 17, 33, 63, 96, 97, 130, 1023, 1024, 1025, 1040, 1089, 2048, 2051, 3000]
    ms = max(lens)
    rng = np.random.default_rng(nser)
    n = len(lens)
    dense, y = np.zeros((n, ms, 5)), np.zeros((n, ms, nser))
    for i, m in enumerate(lens):
        t = knots_of(kind, m, rng)
        dense[i, :m, 0] = t
        for q in range(nser):
            y[i, :m, q] = np.sin(3 * t / t[-1] + q) + 0.1 * np.cos(17 * t / t[-1])
    d, k = torch.tensor(dense, device=dev), torch.tensor(y, device=dev)
    ns = torch.tensor(lens, dtype=torch.int32, device=dev)
    coef = torch.full((n, ms, 4 * nser), 7.0, dtype=torch.float64, device=dev)
    scratch = torch.empty(int(lib().eobhip_spline_scratch_doubles(n, ms)), dtype=torch.float64, device=dev)
    call("eobhip_spline_build_batched", d.data_ptr(), k.data_ptr(), ns.data_ptr(), n, ms, coef.data_ptr(), scratch.data_ptr(),
         P.current_stream())
    got = coef.cpu().numpy()
    for i, m in enumerate(lens):
        assert np.all(got[i, m:] == 7.0)            # nothing past the binary's rows
        assert np.all(got[i, m - 1].reshape(nser, 4)[:, 1:] == 0.0)
        # a backward-stable solve: rounding of the slopes, at most a few hundred ulp on the steepest grading
        assert exact_slopes_error(dense[i, :m, 0], y[i, :m], got[i, :m], nser) < 1e-12


@pytest.mark.parametrize("kind", ["even", "random", "graded", "steep"])
def test_interpolate_TD_chunk_edges(dev, kind):
    lens = [4, 31, 32, 33, 64, 65, 96, 97, 129, 500, 1000]
    n, nsubs, ms = len(lens), 7, max(lens)      # 77 interpolants: more than one group of 64
    rng = np.random.default_rng(9)
    t, y = np.zeros((ms, n)), np.zeros((ms, nsubs, n))
    for i, m in enumerate(lens):
        t[:m, i] = knots_of(kind, m, rng)
        t[m:, i] = t[m - 1, i] + 1.0 + np.arange(ms - m)
        for q in range(nsubs):
            y[:m, q, i] = np.sin(3 * t[:m, i] / t[m - 1, i] + q) + 0.1 * np.cos(17 * t[:m, i] / t[m - 1, i])
    T, Y = torch.tensor(t, device=dev), torch.tensor(y, device=dev)
    B, c1, c2, c3 = (torch.full((ms, nsubs, n), 7.0, dtype=torch.float64, device=dev) for _ in range(4))
    pytdinterp.interpolate_TD_wrap(T, Y, B, c1, c2, c3, torch.tensor(lens, dtype=torch.int32, device=dev), n, nsubs)
    out = [x.cpu().numpy() for x in (c1, c2, c3)]
    b = B.cpu().numpy()
    for i, m in enumerate(lens):
        got = np.zeros((m, 4 * nsubs))
        for q in range(nsubs):
            got[:, 4 * q] = y[:m, q, i]
            for k in range(3):
                got[:, 4 * q + 1 + k] = out[k][:m, q, i]
            assert np.all(b[m:, q, i] == 7.0) and np.all(out[0][m:, q, i] == 7.0)
            assert np.array_equal(b[:m - 1, q, i], out[0][:m - 1, q, i])
            assert out[0][m - 1, q, i] == 0.0
        assert exact_slopes_error(t[:m, i], y[:m, :, i], got, nsubs) < 1e-12
        last = extended_spline(t[:m, i], y[:m, :, i])[3]
        assert np.all(np.abs(b[m - 1, :, i] - last) <= 1e-11 * np.maximum(1.0, np.abs(b[:m, :, i]).max(axis=0)))
