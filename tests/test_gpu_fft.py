"""The library's own real transforms against numpy's, at the edges of their range
of lengths and of the layouts inside it (whole rows in a block, rows as A x B
matrices with A = B and A = 2 B), and the lengths around them that go elsewhere."""
import numpy as np
import pytest
import torch

from eobgpu_amd import pipeline as P

pytestmark = pytest.mark.gpu

EPS = 2.2e-16


@pytest.mark.parametrize("N, rows", [(512, 3), (1024, 17), (2048, 1), (4096, 5), (8192, 3), (1 << 14, 2), (1 << 15, 3), (1 << 16, 1),
                                     (1 << 17, 5), (1 << 18, 2), (1 << 19, 9), (1 << 20, 3), (1 << 21, 2), (1 << 22, 1), (3000, 4)])
def test_rfft_against_numpy(dev, N, rows):
    rng = np.random.default_rng(N + rows)
    h = rng.normal(size=(rows, N))
    h[0] += 3.0 * np.cos(2 * np.pi * 7 * np.arange(N) / N) + 0.5   # a line and an offset
    h[-1, N // 3:] = 0.0
    got = P.rfft_batched(torch.tensor(h, device=dev)).cpu().numpy()
    want = np.fft.rfft(h)
    # a transform's rounding error is at most a few eps log2 N of its 2-norm
    err = np.abs(got - want)
    norm = np.linalg.norm(want, axis=1, keepdims=True)
    assert np.all(np.linalg.norm(err, axis=1, keepdims=True) <= 2 * EPS * np.log2(N) * norm)
    # and in noise it is spread over the bins (row 0's line concentrates it in
    # a few bins, where numpy's own result is 1.2e-10 off an extended-precision one)
    assert np.all((err <= 2 * EPS * np.log2(N) * (np.abs(want) + 8 * norm / np.sqrt(N)))[1:])
    assert np.all(got[:, 0].imag == 0.0) and np.all(got[:, -1].imag == 0.0)


def test_rfft_of_unaligned_and_overlapping_rows(dev):
    """Rows that are 8- but not 16-byte aligned, and an output over its own input, take the general path."""
    N = 4096
    x = torch.randn(2 * N + 1, dtype=torch.float64, device=dev)
    odd = x[1:].view(2, N)
    assert odd.data_ptr() % 16 == 8
    want = np.fft.rfft(odd.cpu().numpy())
    got = P.rfft_batched(odd).cpu().numpy()
    assert np.linalg.norm(got - want) <= 2 * EPS * 12 * np.linalg.norm(want)
    buf = torch.randn(N + 2, dtype=torch.float64, device=dev)
    want = np.fft.rfft(buf[:N].cpu().numpy())
    out = buf.view(torch.complex128).view(1, N // 2 + 1)
    P.rfft_batched(buf[:N].view(1, N), out=out)
    assert np.linalg.norm(out.cpu().numpy()[0] - want) <= 2 * EPS * 12 * np.linalg.norm(want)
