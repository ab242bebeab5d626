"""The right-hand-side, stepper and initial-condition drop-ins on either side of the
batch sizes from which a lane takes a system by itself: the same systems give the
same numbers up to the rounding of the two kernels."""
import numpy as np
import pytest
import torch

from eobgpu_amd import pydopr853, pyEOB
from test_gpu_dropin_blocks import base, run_dropins  # noqa: F401  (base is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [36863, 36864, 43007, 43008, 59391, 59392, 65537])
def test_large_batches_agree_with_the_smallest(dev, base, n):  # noqa: F811
    add, y, h, om, want = base
    got, _ = run_dropins(dev, add, y, h, om, n)
    rep = np.arange(n) % 3
    # the two kernels add the same numbers in the same order; the compiler may fuse other
    # products with their sums: a few ulp of each component, 1e-13 of its size
    for key, w in want.items():
        if key == "err":   # sums that cancel to their last bits: against the step's own scale
            continue
        scale = np.abs(w).max(axis=1, keepdims=True)
        assert np.all(np.abs(got[key] - w[:, rep]) <= 1e-13 * scale), key
        for s in range(3):   # and a system's numbers do not depend on its place
            assert np.all(got[key][:, s::3] == got[key][:, s:s + 1]), key


def test_large_batches_are_no_slower_than_by_blocks(dev, base):  # noqa: F811
    """Four times the systems of a batch that blocks still take: 2.3 times its time with a lane per system, 3.4 by blocks."""
    add0, y0, h0, om, _ = base

    def ms(n):
        rep = np.arange(n) % 3
        T = lambda x: torch.tensor(np.ascontiguousarray(x).reshape(-1), device=dev)  # noqa: E731
        add = add0[:, rep].copy()
        m1, m2, c1, c2 = add[:4]
        eta = m1 * m2 / (m1 + m2) ** 2
        cS, cA = 0.5 * (c1 + c2), 0.5 * (c1 - c2)
        ode = pyEOB.SEOBNRv5Class()
        ode.update_information(T(m1), T(m2), T(eta), T((1 - 2 * eta) * cS + (m1 - m2) / (m1 + m2) * cA), T(cS), T(cA), 1, n, T(add[10:80].T))
        A, Y, x, idx = T(add), T(y0[:, rep]), T(np.zeros(n)), torch.arange(n, dtype=torch.int32, device=dev)
        rhs = torch.zeros(4 * n, dtype=torch.float64, device=dev)
        t = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ode.ODE_Ham_align_AD(x, Y, rhs, A, n, idx)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        return min(t)
    assert ms(131072) < 3.0 * ms(32768)
