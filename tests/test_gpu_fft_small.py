"""Real transforms of few rows: the shapes where the launch takes other block sizes and
pass counts, against numpy, and their time beside the transform library's plans
(which rows at an odd multiple of 8 bytes take)."""
import numpy as np
import pytest
import torch

from eobgpu_amd import pipeline as P
from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu

EPS = 2.2e-16


@pytest.mark.parametrize("N, rows", [(1024, 1), (1024, 2), (1024, 3), (1024, 511), (1024, 1023), (1024, 4097), (2048, 1), (2048, 3),
                                     (2048, 513), (4096, 1), (4096, 257), (8192, 1), (8192, 255), (1 << 14, 1), (1 << 14, 31),
                                     (1 << 14, 32), (1 << 15, 1), (1 << 15, 127), (1 << 15, 128), (1 << 16, 63), (1 << 17, 1),
                                     (1 << 18, 1), (1 << 18, 16), (1 << 19, 1), (1 << 19, 7), (1 << 20, 1), (1 << 20, 4), (1 << 21, 1)])
def test_rfft_of_few_rows(dev, N, rows):
    rng = np.random.default_rng(N + rows)
    h = rng.normal(size=(rows, N))
    got = P.rfft_batched(torch.tensor(h, device=dev)).cpu().numpy()
    want = np.fft.rfft(h)
    err, norm = np.abs(got - want), np.linalg.norm(want, axis=1, keepdims=True)
    # a transform's rounding error is at most a few eps log2 N of its 2-norm, spread over the bins of noise
    assert np.all(np.linalg.norm(err, axis=1, keepdims=True) <= 2 * EPS * np.log2(N) * norm)
    assert np.all(err <= 2 * EPS * np.log2(N) * (np.abs(want) + 8 * norm / np.sqrt(N)))
    assert np.all(got[:, 0].imag == 0.0) and np.all(got[:, -1].imag == 0.0)


@pytest.mark.parametrize("N, rows", [(1 << 10, 1), (1 << 11, 32), (1 << 12, 4), (1 << 14, 1), (1 << 15, 1), (1 << 16, 2), (1 << 18, 1)])
def test_few_rows_take_no_longer_than_a_plan(dev, N, rows):
    st = torch.cuda.current_stream().cuda_stream
    buf = torch.randn(rows * N + 2, dtype=torch.float64, device=dev)
    out = torch.empty((rows, N // 2 + 1), dtype=torch.complex128, device=dev)
    busy = torch.randn(1 << 26, device=dev)

    def us(at):
        def f():
            call("eobhip_rfft_batched", buf.data_ptr() + at, out.data_ptr(), rows, N, st)
        f()
        best = 1e9
        for _ in range(5):
            torch.cuda.synchronize()
            for _ in range(12):
                busy.sin_()       # the launches queue up behind it: the host's time stays out
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(30):
                f()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) / 30 * 1e3)
        return best
    us(8)
    plan, own = us(8), us(0)
    # 0.75 to 1.05 of the plan's time; with one block size for every batch 1.1 to 1.6
    assert own <= (1.25 if N <= 1 << 11 else 1.08) * plan, (own, plan)
