"""The spline builders' rounding: the coefficients' error against extended precision
beside that of the same system eliminated row after row in double precision."""
import numpy as np
import pytest
import torch

from eobgpu_amd import pipeline as P
from eobgpu_amd import pytdinterp
from eobgpu_amd._lib import call
from test_gpu_spline_tiles import extended_spline

pytestmark = pytest.mark.gpu


def serial_spline(t, y):
    """(c1, c2, c3) of the not-a-knot splines of y's columns by one elimination from the first row, a division a step."""
    n, dx = len(t), np.diff(t)
    m = np.diff(y, axis=0) / dx[:, None]
    b, dg, ud, ld = np.zeros_like(y), np.zeros(n), np.zeros(n), np.zeros(n)
    b[1:-1] = 3 * (dx[1:, None] * m[:-1] + dx[:-1, None] * m[1:])
    dg[1:-1], ud[1:-1], ld[1:-1] = 2 * (dx[1:] + dx[:-1]), dx[:-1], dx[1:]
    for i, p, q, u, v in ((0, dx[0], dx[1], m[0], m[1]), (n - 1, dx[-2], dx[-1], m[-2], m[-1])):
        e = p + q
        b[i] = (((p + 2 * e) * q * u + p * p * v) if i == 0 else (q * q * u + (2 * e + q) * p * v)) / e
        dg[i] = q if i == 0 else p
    ud[0], ld[-1] = dx[0] + dx[1], dx[-2] + dx[-1]
    for i in range(1, n):
        w = ld[i] / dg[i - 1]
        dg[i] -= w * ud[i - 1]
        b[i] -= w * b[i - 1]
    s = b / dg[:, None]
    for i in range(n - 2, -1, -1):
        s[i] = (b[i] - ud[i] * s[i + 1]) / dg[i]
    tt = (s[:-1] + s[1:] - 2 * m) / dx[:, None]
    return s[:-1], (m - s[:-1]) / dx[:, None] - tt, tt / dx[:, None]


def test_builders_round_no_worse_than_the_serial_elimination(dev):
    n, rows = 16, 1500
    rng = np.random.default_rng(3)
    t = np.arange(rows) * (0.37 * rng.uniform(0.5, 2, n))[:, None]
    u = (t / t[:, -1:])[:, :, None]
    y = np.sin(rng.uniform(2, 30, (n, 1, 3)) * u + np.arange(3)) + 0.1 * np.cos(17 * u)
    dense = np.zeros((n, rows, 5))
    dense[:, :, 0] = t
    T = lambda a: torch.tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
    ns = torch.full((n,), rows, dtype=torch.int32, device=dev)
    coef = torch.zeros((n, rows, 12), dtype=torch.float64, device=dev)
    d, k = T(dense), T(y)
    call("eobhip_spline_build_batched", d.data_ptr(), k.data_ptr(), ns.data_ptr(), n, rows, coef.data_ptr(), None, P.current_stream())
    B, c1, c2, c3 = (torch.zeros((rows, 3, n), dtype=torch.float64, device=dev) for _ in range(4))
    pytdinterp.interpolate_TD_wrap(T(t.T), T(y.transpose(1, 2, 0)), B, c1, c2, c3, ns, n, 3)
    tile = coef.cpu().numpy().reshape(n, rows, 3, 4)
    drop = [c.cpu().numpy() for c in (c1, c2, c3)]
    sq = np.zeros(3)
    for i in range(n):
        exact, serial = extended_spline(t[i], y[i]), serial_spline(t[i], y[i])
        scale = np.abs(y[i]).max(axis=0) / np.diff(t[i])[:, None] ** np.array([1, 2, 3])[:, None, None]
        for j in range(3):
            for which, c in enumerate((serial[j], tile[i, :-1, :, j + 1], drop[j][:-1, :, i])):
                sq[which] += np.mean((np.abs(c - exact[j]) / scale[j]).astype(float) ** 2)
    rms = np.sqrt(sq)
    # the same roundings, some of them fused: no more than the serial elimination's, to its 1 % of scatter over
    # 200 000 coefficients
    assert rms[1] <= 1.01 * rms[0] and rms[2] <= 1.01 * rms[0], rms / rms[0]
