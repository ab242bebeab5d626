"""The likelihood's second half in one call against the same in stages (resample,
transforms, finish), from the smallest to a large transform size and with every
size of a batch the whole segment's."""
import numpy as np
import pytest
import torch

from eobgpu_amd import configs
from eobgpu_amd import pipeline as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2N,m_min,dt", [(10, 10, 1.0 / 256), (14, 10, 1.0 / 4096), (15, 15, 1.0 / 4096), (18, 10, 1.0 / 8192)])
def test_one_call_likelihood_matches_stages(dev, log2N, m_min, dt):
    N, n = 1 << log2N, 9
    p = configs.small_batch(n=n, seed=17)
    p["r0"] = np.linspace(9.0, 17.0, n)
    M = p["m1"] + p["m2"]
    b = P.EOBBatch(P.make_additional_args(p["m1"], p["m2"], p["chi1"], p["chi2"]), max_step=4096, device=dev)
    b.initial_conditions(p["r0"])
    b.integrate(rtol=1e-10, atol=1e-10, two_pass=True)
    b.hlm22_knots()
    b.build_splines()
    rng = np.random.default_rng(2)
    df = 1.0 / (N * dt)
    data = rng.normal(size=N // 2 + 1) + 1j * rng.normal(size=N // 2 + 1)
    lik = P.SupportLikelihood(data, N, df, m_min_log2=m_min)
    got = []
    for own in (lik._OWN_LOG2, (99, 0)):   # all sizes through the one call, none
        lik._OWN_LOG2 = own
        terms = torch.full((n, 2), np.nan, dtype=torch.float64, device=dev)
        logl = lik(b, M, dt, terms=terms).cpu().numpy()
        got.append((logl, terms.cpu().numpy(), lik.nsamp.cpu().numpy(), lik.mlog2.cpu().numpy()))
    (la, ta, na, ma), (lb, tb, nb, mb) = got
    np.testing.assert_array_equal(na, nb)
    np.testing.assert_array_equal(ma, mb)
    # hh: sums of squares of transforms within log2 N rounding errors of each other; the
    # cross term adds the same products in another order (|sum| <= sum of |h g|)
    h = b.resample_hplus(M, dt, N).cpu().numpy()
    mag = np.abs(h * lik.g.cpu().numpy()[None, :N]).sum(axis=1)
    np.testing.assert_allclose(ta[:, 1], tb[:, 1], rtol=1e-13)
    assert np.all(np.abs(ta[:, 0] - tb[:, 0]) <= 1e-13 * mag)
    assert np.all(np.abs(la - lb) <= 2.0 * df * 1e-13 * (2.0 * mag + tb[:, 1]) + 1e-15 * np.abs(lb))
