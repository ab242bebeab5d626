"""The resampling kernels' sine and cosine against extended precision, over the
decades of their argument and at the edges of its reductions: on the CPU (a host
build of the same source) and on the device, through the resample of a table
whose knots are the samples."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

# half an ulp of the result (5.6e-17 below 1), half of that again for the square of the
# reduced argument in the cosine, and the last terms of the series
BOUND = 1e-16


def arguments(per):
    rng = np.random.default_rng(5)
    x = [10.0 ** rng.uniform(lo, hi, per) for lo, hi in ((-9, 0), (0, 2), (2, 5), (5, 9), (9, 12), (12, 14), (14, 15), (15, 16), (16, 22),
                                                         (22, 100), (100, 308))]
    x.append(rng.integers(1, 1 << 50, per) * (np.pi / 2))                       # near multiples of pi/2
    x.append(2.0 ** rng.integers(44, 1000, per) * rng.integers(1, 1 << 20, per))   # trailing zeros
    e = 2.0 ** np.array([45, 49, 52, 53, 1023])
    # the worst known double for a reduction by pi/2, and the ends of the ranges
    x.append(np.concatenate([e, np.nextafter(e, 0), [0.0, 5e-324, 6381956970095103.0 * 2.0 ** 797, np.finfo(float).max, np.pi / 4, np.pi / 2]]))
    x = np.concatenate(x)
    return np.concatenate([x, -x])


def check(x, s, c):
    X = x.astype(np.longdouble)
    assert np.abs(s - np.sin(X)).max() < BOUND
    assert np.abs(c - np.cos(X)).max() < BOUND


def test_host_build():
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    import tempfile
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "probe.so")
        subprocess.run([cxx, "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-o", out, os.path.join(HERE, "sincos_probe.cpp")], check=True)
        f = ctypes.CDLL(out).probe_sincos_phase
        x = arguments(20000)
        s, c = np.empty_like(x), np.empty_like(x)
        args = [a.ctypes.data_as(ctypes.c_void_p) for a in (x, s, c)]
        f(*args, len(x))
        check(x, s, c)
        x[:3] = np.inf, -np.inf, np.nan
        f(*args, 3)
        assert np.all(np.isnan(s[:3])) and np.all(np.isnan(c[:3]))


@pytest.mark.gpu
@pytest.mark.parametrize("every", [1, 64])   # samples a knot: every row past the staged ones, and staged rows of two
@pytest.mark.parametrize("kind", ["hpc", "modes"])
def test_resampled_phases(dev, every, kind):
    import torch
    from eobgpu_amd._lib import call
    x = arguments(4000)
    x = np.concatenate([[np.inf, -np.inf, np.nan], np.random.default_rng(1).permutation(x)])
    K = 2048
    n, N = -(-len(x) // K), K * every
    arg = np.zeros(n * K)
    arg[:len(x)] = x
    dense, coef = np.zeros((n, K, 5)), np.zeros((n, K, 12))
    dense[:, :, 0] = every * np.arange(K)
    if kind == "hpc":      # h22 = S e^{-2 i phi}; the argument is twice this
        arg = 2 * (arg / 2)
        coef[:, :, 0], coef[:, :, 4] = (arg / 2).reshape(n, K), 1.0
    else:                  # S e^{-i phi}
        coef[:, :, 8], coef[:, :, 0] = arg.reshape(n, K), 1.0
    dv = lambda a, t=torch.float64: torch.as_tensor(a, dtype=t, device=dev)  # noqa: E731
    d, cf, ns, one = dv(dense), dv(coef), dv(np.full(n, K), torch.int32), dv(np.ones(n))
    hp, hc, cnt = dv(np.zeros((n, N))), dv(np.zeros((n, N))), dv(np.zeros(n), torch.int32)
    args = [d.data_ptr(), cf.data_ptr(), ns.data_ptr(), one.data_ptr(), one.data_ptr(), n, K, N]
    if kind == "hpc":
        call("eobhip_resample_hpc", *args, hp.data_ptr(), hc.data_ptr(), cnt.data_ptr(), None)
    else:
        call("eobhip_resample_modes", *args, 1, (ctypes.c_int * 1)(1), hp.data_ptr(), hc.data_ptr(), cnt.data_ptr(), None)
    assert np.all(cnt.cpu().numpy() == every * (K - 1) + 1)
    # all samples of a knot have its phase
    for j in {0, every // 2, every - 1}:
        c, s = (v.view(n, K, every)[:, :K - 1, j].cpu().numpy() for v in (hp, -hc))
        a = arg.reshape(n, K)[:, :K - 1]
        bad = ~np.isfinite(a)
        assert bad.sum() == 3 and np.all(np.isnan(c[bad])) and np.all(np.isnan(s[bad]))
        check(a[~bad], s[~bad], c[~bad])
