"""What a served binary is said to take of device memory is what its pool allocates
for it, and is what the passes use."""
import torch

from eobgpu_amd._lib import lib
from eobgpu_amd.serving import SlotPool


def test_bytes_per_binary_are_the_buffers():
    c, ms, N = 3, 96, 256
    pool = SlotPool(c, ms, N, device="cpu")
    held = sum(v.numel() * v.element_size() for v in vars(pool).values() if isinstance(v, torch.Tensor))
    assert held == c * pool.bytes_per_binary()
    # tables, trajectory rows, three knot series and their coefficients, samples, bins, and the results
    tables = int(lib().eobhip_bindata_bytes()) + int(lib().eobhip_modes_bytes())
    assert pool.bytes_per_binary() == tables + 8 * ms * (5 + 3 + 12) + 8 * N + 16 * (N // 2 + 1) + 4 * 4 + 2 * 8
