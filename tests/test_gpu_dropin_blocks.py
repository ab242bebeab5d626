"""The reference's right-hand-side, stepper and initial-condition drop-ins at the
batch sizes where the systems per block change and the last block is ragged: a
system's numbers do not depend on the batch it is in (they are the same bits),
and in the smallest batch they are the oracle's."""
import numpy as np
import pytest
import torch

from eobgpu_amd import configs, pipeline as P, pydopr853, pyEOB

pytestmark = pytest.mark.gpu


def run_dropins(dev, add, y, h, om, n):
    """every drop-in on n systems, system i being base system i mod len(h)"""
    rep = np.arange(n) % len(h)
    add, y, h, om = add[:, rep].copy(), y[:, rep], h[rep], om[rep]
    add[4] = om

    def T(x):
        return torch.tensor(np.ascontiguousarray(x, dtype=np.float64).reshape(-1), device=dev)
    m1, m2, c1, c2 = add[:4]
    eta = m1 * m2 / (m1 + m2) ** 2
    cS, cA = 0.5 * (c1 + c2), 0.5 * (c1 - c2)
    ode = pyEOB.SEOBNRv5Class()
    ode.update_information(T(m1), T(m2), T(eta), T((1 - 2 * eta) * cS + (m1 - m2) / (m1 + m2) * cA), T(cS), T(cA), 1, n, T(add[10:80].T))
    A, Y, H, x, idx = T(add), T(y), T(h), T(np.zeros(n)), torch.arange(n, dtype=torch.int32, device=dev)
    z = lambda m: torch.zeros(m, dtype=torch.float64, device=dev)  # noqa: E731
    rhs, ks = z(4 * n), [z(4 * n) for _ in range(10)]
    ode.ODE_Ham_align_AD(x, Y, rhs, A, n, idx)
    pydopr853.dormandPrinceSteps(x, z(n), Y, H, z(4 * n), A, *ks, z(4 * n), 4, n, 80, ode, idx)
    err, new = z(n), z(4 * n)
    pydopr853.error(err, Y, new, H, ks[0], ks[1], ks[2], *ks[5:10], n, 4)
    rg = om ** (-2.0 / 3)
    xo, args, pr = z(2 * n), z(4 * n), z(n)
    pyEOB.root_find_all(xo, T(np.array([rg, np.sqrt(rg)])), args, A, 1000, 1e-12, n, 2, 4, 80)
    args.view(4, n)[0], args.view(4, n)[3] = xo[:n], xo[n:]
    ode.root_find_scalar_all(pr, T(np.array([np.full(n, -3e-2), np.zeros(n)])), args, A, 1000, 1e-12, n, 4, 80)
    out = {"rhs": rhs.view(4, n), "new": new.view(4, n), "err": err.view(1, n), "x": xo.view(2, n), "pr": pr.view(1, n)}
    out.update({"k%d" % i: k.view(4, n) for i, k in enumerate(ks)})
    return {k: v.cpu().numpy() for k, v in out.items()}, add


@pytest.fixture(scope="module")
def base(dev, oracle):
    p = configs.uneven_batch(n=3, seed=12)
    add = P.make_additional_args(p["m1"], p["m2"], p["chi1"], p["chi2"])
    rng = np.random.default_rng(4)
    r = np.array([9.0, 17.0, 33.0])
    y = np.array([r, rng.uniform(0, 50, 3), -1e-3 * (10.0 / r) ** 3, np.sqrt(r) * (1 + 1.5 / r)])
    h, om = 0.5 * r ** 1.5, 20.0 * np.pi * (p["m1"] + p["m2"]) * P.MTSUN_SI
    out, add3 = run_dropins(dev, add, y, h, om, 3)
    co = oracle.fac_coeffs(add3)
    assert np.allclose(out["rhs"], oracle.rhs(y, add3, co), rtol=5e-10, atol=1e-14)
    assert np.array_equal(out["rhs"], out["k0"])     # the stepper's first stage is the right-hand side
    return add, y, h, om, out


@pytest.mark.parametrize("n", [1, 2, 4, 5, 63, 1024, 1025, 4099, 16384, 17001])
def test_results_do_not_depend_on_the_batch(dev, base, n):
    add, y, h, om, want = base
    got, _ = run_dropins(dev, add, y, h, om, n)
    rep = np.arange(n) % 3
    for key, w in want.items():
        assert np.array_equal(got[key], w[:, rep]), key
