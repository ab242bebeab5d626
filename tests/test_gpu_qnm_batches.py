"""Kerr QNMs in batches whose roots are shared out differently: by groups of lanes, by
lanes, and both in one call (spins and modes with and without a table)."""
import numpy as np
import pytest
import torch

from eobgpu_amd import eobstuff as ES
from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu


def qnm(l, m, af):
    return np.asarray(ES.compute_QNM(l, m, 0, af, np.ones(len(af))))


@pytest.mark.parametrize("l,m", [(2, 2), (3, 3), (2, -2)])
@pytest.mark.parametrize("n", [1, 5, 63, 65, 49152, 49153])
def test_roots_do_not_depend_on_the_batch(dev, l, m, n):
    base = np.array([0.3, -0.6, 0.9905, 0.7, -0.95, 0.0, 0.985, 0.99])   # one past the table
    one = np.array([qnm(l, m, base[i:i + 1])[0] for i in range(len(base))])
    assert len(set(one)) == len(base) and np.all(one.real > 0) and np.all(one.imag < 0)
    at = np.arange(n) % len(base)
    # groups and lanes round differently: both are within 1e-14 of the root
    assert np.abs(qnm(l, m, base[at]) - one[at]).max() <= 2e-14 * np.abs(one).max()


def test_many_roots_without_a_table_keep_the_chip_busy(dev):
    """Sixteen times the roots, all on the spin path: the chip still has lanes for them, so a lane per root takes little longer."""
    def ms(n):
        af, out = torch.full((n,), 0.3, dtype=torch.float64, device=dev), torch.empty(2 * n, dtype=torch.float64, device=dev)
        t = []
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            call("eobhip_kerr_qnm", 2, -2, af.data_ptr(), n, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        return min(t)
    assert ms(65536) < 2.0 * ms(4096)
