"""Uniform resampling where rows of 128 samples meet few, many and no knots and
where templates end at the edges of rows and runs, against numpy."""
import ctypes

import numpy as np
import pytest
import torch
from scipy.interpolate import CubicSpline

from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu


def knots_of(kind, rng):
    if kind == "wide":      # several rows to an interval, then a fixed-step tail of many knots a row
        d = np.concatenate([np.full(20, 300.0), np.full(300, 0.7), np.full(5, 300.0)])
    elif kind == "few":     # 1 to 9 knots a row
        d = np.concatenate([np.full(20, 128.0 / k) for k in range(1, 10)])
    elif kind == "lanes":   # 63, 64 and 65 knots a row, then every sample its own knot, then one interval
        d = np.concatenate([np.full(300, 128.0 / k) for k in (63, 64, 65, 128, 300)] + [np.full(1, 2000.0)])
    else:
        d = rng.uniform(0.01, 1.0, 3000) * rng.choice([0.1, 10.0], 3000)
    return 3.0 + np.concatenate([[0.0], np.cumsum(d)])


@pytest.mark.parametrize("kind", ["wide", "few", "lanes", "random"])
@pytest.mark.parametrize("ms", [(2,), (2, 1, 3), (2, 1, 3, 4, 5)])
def test_resample_rows(dev, kind, ms):
    rng = np.random.default_rng(len(ms))
    t = knots_of(kind, rng)
    full = len(t)
    # the whole table and templates that end just before, at and after row and run edges
    ends = [t[-1] - 3.0] + [k + e for k in (128, 1024) for e in (-0.5, 0.0, 0.5)] + [0.5]
    lens = [full] + [max(2, int(np.searchsorted(t, 3.0 + e, "right"))) for e in ends[1:]] + [1]
    n, nm = len(lens), len(ms)
    dTs = np.where(np.arange(n) % 2, 1.0, 0.75)
    N = int((t[-1] - 3.0) * 0.8) | 1   # odd: every other row starts 8 bytes off; the first template is cut
    phi = 0.15 * t + 2.0 * np.sin(t / 60.0)
    series = [np.cos(t / (30.0 + 7 * q)) + 1.5 for q in range(2 * nm)] + [phi]
    dense = np.zeros((n, full, 5))
    dense[:, :, 0] = t
    coef = np.zeros((n, full, 2 * nm + 1, 4))
    for q, y in enumerate(series):
        c = CubicSpline(t, y).c[::-1]
        coef[:, :-1, q] = c.T
        coef[:, -1, q, 0] = y[-1]   # the last knot's row: its value
    amp = np.linspace(0.5, 2.0, n)
    dv = lambda a, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)
    want = np.zeros((n, N), complex)
    counts = np.zeros(n, int)
    for b in range(n):
        if lens[b] < 2:
            continue
        tb = t[:lens[b]]
        counts[b] = min(N, int((tb[-1] - tb[0]) / dTs[b]) + 1)
        tj = tb[0] + np.arange(counts[b]) * dTs[b]
        i = np.maximum(np.searchsorted(tb, tj, "right") - 1, 0)
        x = (tj - tb[i])[:, None]
        v = coef[b, i, :, 0] + x * (coef[b, i, :, 1] + x * (coef[b, i, :, 2] + x * coef[b, i, :, 3]))
        for q, m in enumerate(ms):
            want[b, :counts[b]] += amp[b] * (v[:, q] + 1j * v[:, nm + q]) * np.exp(-1j * m * v[:, 2 * nm])
    # times are below 2^13 (half an ulp 4.5e-13) and m dphi/dt below 1; m phi is below
    # 2^13 and is formed by m products: 5e-12 per unit of |S| covers each
    bound = 5e-12 * 2.5 * np.sqrt(2.0) * nm * amp.max()
    assert t[-1] < 2 ** 13 and max(ms) * phi.max() < 2 ** 13

    def check(hp, hc, ns):
        np.testing.assert_array_equal(ns.cpu().numpy(), counts)
        assert np.abs(hp.cpu().numpy() - want.real).max() < bound
        if hc is not None:
            assert np.abs(hc.cpu().numpy() - want.imag).max() < bound

    hp, hc = torch.full((n, N), 9.0, dtype=torch.float64, device=dev), torch.full((n, N), 9.0, dtype=torch.float64, device=dev)
    ns = torch.zeros(n, dtype=torch.int32, device=dev)
    d, ln, a, dT = dv(dense), dv(lens, torch.int32), dv(amp), dv(dTs)
    c = dv(coef)
    mm = (ctypes.c_int * nm)(*ms)
    call("eobhip_resample_modes", d.data_ptr(), c.data_ptr(), ln.data_ptr(), a.data_ptr(), dT.data_ptr(), n, full, N, nm, mm, hp.data_ptr(),
         hc.data_ptr(), ns.data_ptr(), None)
    check(hp, hc, ns)
    if ms == (2,):
        # the (2,2) tables hold phi first
        c22 = dv(coef[:, :, [2, 0, 1]])
        hp.fill_(9.0)
        hc.fill_(9.0)
        ns.zero_()
        call("eobhip_resample_hpc", d.data_ptr(), c22.data_ptr(), ln.data_ptr(), a.data_ptr(), dT.data_ptr(), n, full, N, hp.data_ptr(),
             hc.data_ptr(), ns.data_ptr(), None)
        check(hp, hc, ns)
        hp.fill_(9.0)
        call("eobhip_resample_hplus", d.data_ptr(), c22.data_ptr(), ln.data_ptr(), a.data_ptr(), dT.data_ptr(), n, full, N, hp.data_ptr(),
             ns.data_ptr(), None)
        check(hp, None, ns)
