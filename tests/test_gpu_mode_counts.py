"""The mode sum of 6 to 15 modes, every m
up to 8, repeated and in any order, against numpy: knots that several rows of 128
samples share, that one row passes in tens and that it passes in hundreds."""
import ctypes

import numpy as np
import pytest
import torch

from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu

MS = {6: (5, 1, 8, 3, 3, 2), 8: (2, 1, 3, 4, 5, 2, 3, 6), 15: (8, 2, 7, 7, 1, 3, 6, 4, 5, 8, 2, 1, 3, 3, 4)}


@pytest.mark.parametrize("nm", sorted(MS))
def test_many_modes(dev, nm):
    ms = MS[nm]
    assert len(ms) == nm
    rng = np.random.default_rng(nm)
    t = 3.0 + np.concatenate([[0.0], np.cumsum(np.concatenate([np.full(6, 300.0), rng.uniform(1.0, 20.0, 100), np.full(800, 0.3),
                                                                [400.0]]))])
    K = len(t)
    lens = np.array([K, K - 1, 200, 3, 1, 0])
    n, N, dT, amp = len(lens), 3001, 1.0, np.linspace(0.5, 2.0, len(lens))   # odd: every other row starts 8 bytes off
    phi = 0.1 * t + np.sin(t / 60.0)
    x = rng.normal(size=(n, K, 2 * nm + 1, 4))
    coef = x * np.array([1.0, 1e-3, 1e-6, 1e-9])
    coef[:, :, 2 * nm, 0], coef[:, :, 2 * nm, 1:] = phi, [0.1, 1e-7, 1e-11]
    dense = np.zeros((n, K, 5))
    dense[:, :, 0] = t
    want, size, counts = np.zeros((n, N), complex), 0.0, np.zeros(n, int)
    for b in range(n):
        if lens[b] < 2:
            continue
        tb = t[:lens[b]]
        counts[b] = min(N, int((tb[-1] - tb[0]) / dT) + 1)
        tj = tb[0] + np.arange(counts[b]) * dT
        i = np.searchsorted(tb, tj, "right") - 1
        d = (tj - tb[i])[:, None]
        v = coef[b, i, :, 0] + d * (coef[b, i, :, 1] + d * (coef[b, i, :, 2] + d * coef[b, i, :, 3]))
        for q, m in enumerate(ms):
            want[b, :counts[b]] += amp[b] * (v[:, q] + 1j * v[:, nm + q]) * np.exp(-1j * m * v[:, 2 * nm])
        size = max(size, amp[b] * np.abs(v[:, :2 * nm]).sum(axis=1).max())
    # times below 2^12 (an ulp 9e-13 of argument, of slopes below 1) and m phi below 2^13, formed by
    # m products: 5e-12 of the sum of the amplitudes covers both
    assert t[-1] < 2 ** 12 and max(ms) * phi.max() < 2 ** 13
    dv = lambda a, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)  # noqa: E731
    d, c, ln, a, dt = dv(dense), dv(coef), dv(lens, torch.int32), dv(amp), dv(np.full(n, dT))
    hp, hc = (torch.full((n, N), 9.0, dtype=torch.float64, device=dev) for _ in range(2))
    ns = torch.zeros(n, dtype=torch.int32, device=dev)
    call("eobhip_resample_modes", d.data_ptr(), c.data_ptr(), ln.data_ptr(), a.data_ptr(), dt.data_ptr(), n, K, N, nm, (ctypes.c_int * nm)(*ms),
         hp.data_ptr(), hc.data_ptr(), ns.data_ptr(), None)
    np.testing.assert_array_equal(ns.cpu().numpy(), counts)
    got = (hp + 1j * hc).cpu().numpy()
    assert np.abs(got - want).max() < 5e-12 * size
    assert not got[np.arange(N)[None, :] >= counts[:, None]].any()
