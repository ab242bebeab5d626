"""The merger-ringdown template's ringdown samples, which blocks of their own write:
series of every length around the attachment and the ringdown's end, where the two
kinds of blocks meet at odd and even samples, are prefixes of one long series."""
import ctypes

import numpy as np
import pytest
import torch

from eobgpu_amd import configs
from eobgpu_amd import pipeline as P
from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes", [((2, 2),), P.REFERENCE_MODES + ((2, 2), (3, 3))])
def test_series_meet_at_the_attachment(dev, modes):
    n, dt = 4, 1.0 / 16384
    p = configs.small_batch(n=n, seed=31)
    b = P.EOBBatch(P.make_additional_args(p["m1"], p["m2"], p["chi1"], p["chi2"]), max_step=4096, device=dev)
    b.initial_conditions(np.array([10.5, 10.4, 10.3, 8.0]))
    b.integrate(rtol=1e-10, atol=1e-10, two_pass=True)
    b.num_steps[3] = 3                        # a failed binary: no samples
    M = p["m1"] + p["m2"]
    b.hlm_modes_knots(modes)
    b.build_mode_splines()
    q = b.imr_params(M, dt)
    ls, ms = ((ctypes.c_int * len(modes))(*[lm[k] for lm in modes]) for k in (0, 1))
    amp = torch.tensor([1.0, -2.0, 0.5, 1.0], dtype=torch.float64, device=dev)

    def template(N):
        hp, hc = (torch.full((n, N), 9.0, dtype=torch.float64, device=dev) for _ in range(2))
        ns = torch.full((n,), -5, dtype=torch.int32, device=dev)
        call("eobhip_imr_resample", b.dense.data_ptr(), b.num_steps.data_ptr(), b.mode_coef.data_ptr(), b.rp_coef.data_ptr(),
             amp.data_ptr(), q["dT_M"].data_ptr(), n, b.max_step, N, len(modes), ls, ms, q["nqc"].data_ptr(), q["rd"].data_ptr(),
             q["binf"].data_ptr(), q["bini"].data_ptr(), hp.data_ptr(), hc.data_ptr(), ns.data_ptr(), P.current_stream())
        return (hp + 1j * hc).cpu().numpy(), ns.cpu().numpy()

    idx, nadd = (q["bini"].cpu().numpy()[:3, k].astype(int) for k in (1, 2))
    end = idx + nadd
    assert len({int(i) % 2 for i in idx}) == 2      # odd and even attachments
    full, ns = template(int(end.max()) + 3000)
    assert np.array_equal(ns[:3], end) and ns[3] == 0
    for i in range(3):
        assert np.all(full[i, :end[i]] != 0.0) and np.all(np.isfinite(full[i])) and not full[i, end[i]:].any()
        assert np.abs(full[i, :end[i]]).max() < 9.0
        # neighbours across the attachment are as close as the samples around them
        step = np.abs(np.diff(full[i]))
        assert step[idx[i]] < 2.0 * step[idx[i] - 40:idx[i] + 40].max()
    assert not full[3].any()
    turns = {N for k in range(4, full.shape[1] // 512, 8) for N in (512 * k, 512 * k - 5)}      # grids whose rows take turns
    assert max(turns) > idx.min()
    for N in sorted({int(v) + e for v in np.concatenate([idx, end]) for e in (-1, 0, 1, 2, 3)} | {1, 2, 129} | turns):
        h, ns = template(N)
        assert np.array_equal(h, full[:, :N]), N
        assert np.array_equal(ns[:3], np.minimum(end, N)) and ns[3] == 0


def test_ringdowns_of_a_grid_of_eight(dev):
    """512 binaries of 2^13 samples (eight blocks each, four of them the ringdown's) against 17 runs each (nine)."""
    n = 512
    p = configs.uneven_batch(n=n, seed=4)
    b = P.EOBBatch.from_params(p["m1"], p["m2"], p["chi1"], p["chi2"])
    b.initial_conditions(p["r0"])
    b.integrate(rtol=1e-10, atol=1e-10)
    b.hlm_modes_knots(P.REFERENCE_MODES)
    b.build_mode_splines()
    M, dt = p["m1"] + p["m2"], 1.0 / 16384
    q = b.imr_params(M, dt)

    def best(N):
        times = []
        for _ in range(10):
            s, e = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            torch.cuda.synchronize()
            big.sin_()   # the launches are made meanwhile
            s.record()
            for _ in range(4):
                call("eobhip_imr_resample", *args[0], n, b.max_step, N, *args[1], P.current_stream())
            e.record()
            torch.cuda.synchronize()
            times.append(s.elapsed_time(e))
        return min(times)

    big = torch.randn(1 << 28, device=dev)
    hp, hc = (torch.empty(n * 9000, dtype=torch.float64, device=dev) for _ in range(2))
    amp, ns = torch.ones(n, dtype=torch.float64, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    ls, ms = ((ctypes.c_int * 5)(*[lm[k] for lm in P.REFERENCE_MODES]) for k in (0, 1))
    args = ([x.data_ptr() for x in (b.dense, b.num_steps, b.mode_coef, b.rp_coef, amp, q["dT_M"])],
            [5, ls, ms] + [x.data_ptr() for x in (q["nqc"], q["rd"], q["binf"], q["bini"], hp, hc, ns)])
    # 6 % fewer samples; with every ringdown on the same four of the eight XCDs 1.6 times as long
    assert best(8192) < 1.25 * best(8704)
