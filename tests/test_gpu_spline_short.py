"""The (2,2) spline builder on series too short for a not-a-knot spline: 0, 1 and 2 rows
(values, no slopes), 3 rows (whose system has no single solution: values, and
pieces that meet the next knot if they are finite), beside ordinary ones."""
import numpy as np
import pytest
import torch

from eobgpu_amd import pipeline as P
from eobgpu_amd._lib import call

pytestmark = pytest.mark.gpu


def test_short_series(dev):
    lens = [0, 1, 2, 3, 40, 2, 0, 3, 1100, 1]
    n, ms = len(lens), 1200
    rng = np.random.default_rng(2)
    dense, y = rng.normal(size=(n, ms, 5)), rng.normal(size=(n, ms, 3))
    dense[:, :, 0] = np.cumsum(rng.uniform(0.5, 2.0, (n, ms)), axis=1)
    d, k, ns = torch.tensor(dense, device=dev), torch.tensor(y, device=dev), torch.tensor(lens, dtype=torch.int32, device=dev)
    coef = torch.full((n, ms, 12), 7.0, dtype=torch.float64, device=dev)
    call("eobhip_spline_build_batched", d.data_ptr(), k.data_ptr(), ns.data_ptr(), n, ms, coef.data_ptr(), None, P.current_stream())
    c = coef.cpu().numpy().reshape(n, ms, 3, 4)
    for b, m in enumerate(lens):
        assert np.all(c[b, m:] == 7.0)
        assert np.array_equal(c[b, :m, :, 0], y[b, :m])
        if m <= 2:
            assert not c[b, :m, :, 1:].any()
            continue
        assert not c[b, m - 1, :, 1:].any()
        h = np.diff(dense[b, :m, 0])[:, None]
        a = c[b, :m - 1]
        terms = [a[..., 0], a[..., 1] * h, a[..., 2] * h ** 2, a[..., 3] * h ** 3]
        end, size = sum(terms), sum(np.abs(t) for t in terms)
        ok = np.isfinite(size)
        assert m == 3 or ok.all()
        assert np.all(np.abs(end - y[b, 1:m])[ok] <= 1e-14 * size[ok])
