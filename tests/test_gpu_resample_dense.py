"""Resampling of tables with 0.3 to 700 knots a row of 128 samples (less, as many and more
than a wavefront stages, compares and holds), in runs of one row and of four, with
phases beyond 2^49, against numpy; the inspirals of merger-ringdown templates at 1 / k of
their rate against every k-th sample."""
import ctypes

import numpy as np
import pytest
import torch

from eobgpu_amd import configs
from eobgpu_amd import pipeline as P
from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu

DENSITIES = (0.3, 1, 7, 8, 9, 10, 15, 16, 17, 27, 28, 29, 61, 62, 63, 64, 65, 130, 700)
ROWS = 9.4   # of 128 samples in a template


def table(S):
    """Knot times, coefficients of S series and phi (series S) of one binary per density, and of one
    with all of them in turn; every other one's phase past 2^49 in a part of it."""
    rng = np.random.default_rng(S)
    gap = [np.concatenate([rng.uniform(0.2, 1.8, int(np.ceil(ROWS * d))) * 128 / d]) for d in DENSITIES]
    gap.append(np.concatenate([rng.uniform(0.2, 1.8, max(1, int(d))) * 128 / d for d in DENSITIES]))
    lens = np.array([len(g) + 1 for g in gap])
    n, K = len(gap), lens.max()
    dense, coef = np.zeros((n, K, 5)), np.zeros((n, K, S + 1, 4))
    for b, g in enumerate(gap):
        t = 5.0 + np.concatenate([[0.0], np.cumsum(g)])
        dense[b, :lens[b], 0] = t
        coef[b, :lens[b], :S] = rng.normal(size=(lens[b], S, 4)) * np.array([1.0, 1e-3, 1e-6, 1e-9])
        coef[b, :lens[b], S] = np.stack([0.1 * t + np.sin(t / 60.0), np.full(lens[b], 0.1), np.full(lens[b], 1e-7), np.full(lens[b], 1e-11)], axis=1)
        if b % 2:   # whole numbers, m times which are exact
            far = (t > 400.0) & (t < 600.0)
            coef[b, :lens[b]][far, S] = np.stack([2.0 ** 49 + np.floor(t[far] * 16), 0 * t[far], 0 * t[far], 0 * t[far]], axis=1)
    return dense, coef, lens


def sampled(dense, coef, lens, N, dT):
    """(values of every series [count, S + 1], count) of each binary."""
    out = []
    for b in range(len(lens)):
        t = dense[b, :lens[b], 0]
        count = min(N, int((t[-1] - t[0]) / dT) + 1)
        tj = t[0] + np.arange(count) * dT
        i = np.searchsorted(t, tj, "right") - 1
        d = (tj - t[i])[:, None]
        out.append(coef[b, i, :, 0] + d * (coef[b, i, :, 1] + d * (coef[b, i, :, 2] + d * coef[b, i, :, 3])))
    return out


@pytest.mark.parametrize("nm", [0, 1, 5, 15])   # 0: the (2, 2) build
@pytest.mark.parametrize("N", [1000, 1301, 53377])   # 20 binaries: runs of one row, of one, of four
def test_rows_of_many_knots(dev, nm, N):
    ms = (2,) if nm == 0 else (2, 8, 1, 3, 5, 4, 2, 7, 6, 1, 8, 3, 3, 2, 5)[:nm]
    S = 2 * len(ms)
    dense, coef, lens = table(S)
    n, K, dT, amp = len(lens), dense.shape[1], 1.0, np.linspace(0.5, 2.0, len(lens))
    want, size, counts = np.zeros((n, N), complex), 0.0, np.zeros(n, int)
    for b, v in enumerate(sampled(dense, coef, lens, N, dT)):
        counts[b] = len(v)
        for q, m in enumerate(ms):
            want[b, :counts[b]] += amp[b] * (v[:, q] + 1j * v[:, len(ms) + q]) * np.exp(-1j * (m * v[:, S]))
        size = max(size, amp[b] * np.abs(v[:, :S]).sum(axis=1).max())
    # times below 2^12 (an ulp 9e-13 of argument, of slopes below 1) and, but where they are whole
    # numbers, m phi below 2^13, formed by m products: 5e-12 of the sum of the amplitudes covers both
    assert dense[:, :, 0].max() < 2 ** 12 and counts.min() > 500 and (N * n < 128 * 8192) == (N < 5000)
    dv = lambda a, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)  # noqa: E731
    c = coef if nm else np.stack([coef[:, :, 2], coef[:, :, 0], coef[:, :, 1]], axis=2)
    d, c, ln, a, dt = dv(dense), dv(c), dv(lens, torch.int32), dv(amp), dv(np.full(n, dT))
    hp, hc = (torch.full((n, N), 9.0, dtype=torch.float64, device=dev) for _ in range(2))
    ns = torch.zeros(n, dtype=torch.int32, device=dev)
    if nm:
        call("eobhip_resample_modes", d.data_ptr(), c.data_ptr(), ln.data_ptr(), a.data_ptr(), dt.data_ptr(), n, K, N, nm,
             (ctypes.c_int * nm)(*ms), hp.data_ptr(), hc.data_ptr(), ns.data_ptr(), None)
    else:
        call("eobhip_resample_hpc", d.data_ptr(), c.data_ptr(), ln.data_ptr(), a.data_ptr(), dt.data_ptr(), n, K, N, hp.data_ptr(),
             hc.data_ptr(), ns.data_ptr(), None)
    np.testing.assert_array_equal(ns.cpu().numpy(), counts)
    got = (hp + 1j * hc).cpu().numpy()
    assert np.abs(got - want).max() < 5e-12 * size
    assert not got[np.arange(N)[None, :] >= counts[:, None]].any()
    if nm == 0:   # h+ alone is the same
        call("eobhip_resample_hplus", d.data_ptr(), c.data_ptr(), ln.data_ptr(), a.data_ptr(), dt.data_ptr(), n, K, N, hc.data_ptr(),
             ns.data_ptr(), None)
        assert torch.equal(hc, hp)


@pytest.mark.parametrize("modes", [((2, 2),), ((2, 2), (2, 1), (3, 3), (4, 4), (5, 5)),
                                   ((2, 2), (2, 1), (3, 3), (4, 4), (5, 5), (2, 2), (2, 1), (3, 3))])
def test_inspirals_of_few_samples(dev, modes):
    p = configs.small_batch(n=3, seed=31)
    b = P.EOBBatch(P.make_additional_args(p["m1"], p["m2"], p["chi1"], p["chi2"]), max_step=4096, device=dev)
    b.initial_conditions(np.full(3, 10.5))
    b.integrate(rtol=1e-10, atol=1e-10, two_pass=True)
    b.hlm_modes_knots(modes)
    b.build_mode_splines()
    q, n, nm = b.imr_params(p["m1"] + p["m2"], 1.0 / 16384), 3, len(modes)
    amp = torch.ones(n, dtype=torch.float64, device=dev)
    arr = lambda i: (ctypes.c_int * nm)(*[lm[i] for lm in modes])  # noqa: E731

    def inspiral(k, N):
        bini, dT = q["bini"].clone(), q["dT_M"] * k
        bini[:, 1] = bini[:, 1] // k
        hp, hc = (torch.full((n, N), 9.0, dtype=torch.float64, device=dev) for _ in range(2))
        ns = torch.zeros(n, dtype=torch.int32, device=dev)
        call("eobhip_imr_resample", b.dense.data_ptr(), b.num_steps.data_ptr(), b.mode_coef.data_ptr(), b.rp_coef.data_ptr(), amp.data_ptr(),
             dT.data_ptr(), n, b.max_step, N, nm, arr(0), arr(1), q["nqc"].data_ptr(), q["rd"].data_ptr(), q["binf"].data_ptr(),
             bini.data_ptr(), hp.data_ptr(), hc.data_ptr(), ns.data_ptr(), None)
        return (hp + 1j * hc).cpu().numpy(), bini[:, 1].cpu().numpy()

    fine, last = inspiral(1, 1 << 19)   # runs of four rows
    assert (last < 1 << 19).all()
    scale = np.abs(fine).max()
    for k in (1, 2, 4, 16, 64, 256, 1024):
        for N in (4097, 1 << 19):
            h, top = inspiral(k, N)
            for i in range(n):
                m = min(N, top[i] + 1)
                # the same times (k is a power of two); each mode is a few dozen operations on
                # phases below 2^12 (an ulp 9e-13, times m)
                assert np.abs(h[i, :m] - fine[i, :k * m:k][:m]).max() < 1e-11 * scale


@pytest.mark.parametrize("nm", [1, 5])
def test_rows_of_many_knots_are_not_gathered_one_by_one(dev, nm):
    """4096 binaries x 4096 samples with 17 knots a row against the same with two in three rows: the
    tables are as many bytes as the series for one mode and three times as many for five."""
    n, N, room = 4096, 4096, 512
    cm = 1e-3 * torch.randn(n, room, 4 * (2 * nm + 1), dtype=torch.float64, device=dev)
    a = torch.ones(n, dtype=torch.float64, device=dev)
    hp, hc = (torch.empty(n, N, dtype=torch.float64, device=dev) for _ in range(2))
    ns = torch.zeros(n, dtype=torch.int32, device=dev)

    def best(K):
        d = torch.zeros(n, room, 5, dtype=torch.float64, device=dev)
        d[:, :, 0] = torch.arange(room, device=dev) * (N / K)
        ln, dT = torch.full((n,), K, dtype=torch.int32, device=dev), 1.1 * a
        times = []
        for _ in range(8):
            s, e = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            s.record()
            for _ in range(4):
                call("eobhip_resample_modes", d.data_ptr(), cm.data_ptr(), ln.data_ptr(), a.data_ptr(), dT.data_ptr(), n, room, N, nm,
                     (ctypes.c_int * nm)(*range(1, nm + 1)), hp.data_ptr(), hc.data_ptr(), ns.data_ptr(), torch.cuda.current_stream().cuda_stream)
            e.record()
            torch.cuda.synchronize()
            times.append(s.elapsed_time(e))
        return min(times)

    # 1.9 and 2.3 as measured; gathered from memory, a lane's two samples in turn, 3.7 and 4.8
    assert best(500) < 3.0 * best(20)
