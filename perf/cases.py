"""The work that a user of this framework has it do, as cases that can be timed.

``listed()`` are the cases; ``draw(rng)`` gives one more of the same ranges;
``prepare(case, seed)`` makes what a program has in hand before the call,
``run(state)`` is one pass through the public entry points, ``work(case)`` the
bytes and operations that the path cannot do without and ``exact(case, seed)``
the same outputs from plain torch in 64 bits, where they have such a value.

Kinds of case:

  step        one attempted step of the reference's host loop: the drop-ins
              ``dormandPrinceSteps``, ``error`` and ``controllerSuccess``
  ic          the reference's initial-condition solvers as drop-ins
  trajectory  tables, circular start and the two-pass adaptive trajectory
  splines     not-a-knot splines of long chirps (thousands of knots each)
  modes       higher modes on the knots, their splines and the mode sum
  imr         the same modes with the merger-ringdown attachment
  likelihood  many templates against one data set, from each one's support
  direct      the same through (2,2) knots, splines, full-length transforms
  detector    polarizations, their transforms, interferometers' signals
  dropin      the reference's template path as drop-ins: ``interpolate_TD_wrap``,
              ``TDInterp_wrap2``, transforms, ``all_in_one_likelihood``
  pass        the whole streamed pass over a batch of proposals

All binaries are drawn as ``configs.uneven_batch`` draws them (q ~ U[1,10],
log10 M ~ U[1,2], chi ~ U[-0.9,0.9], r0 ~ U[15,40]) from the seed.
"""
import math

import numpy as np
import torch

from eobgpu_amd import configs, detector, pipeline, pydopr853, pyEOB, pytdinterp

MTSUN = pipeline.MTSUN_SI
F0 = 200.0   # corner of the analytic noise curve
MODES = ((2, 2), (2, 1), (3, 3), (4, 4), (5, 5), (3, 2), (4, 3), (6, 6))
STEP_FLOPS = 50663      # FP64 operations of one attempted step
RHS_FLOPS = 4120
ATTEMPTS = 775          # mean attempted steps of a binary of these batches at 1e-10
KNOTS = 600             # mean knots of one


def listed():
    return [
        # the reference's driver on its smallest batch: three synchronous calls per attempted step, all latency
        {"name": "step_16", "kind": "step", "n": 16},
        # the start of a proposal batch through the reference's own solvers
        {"name": "ic_1024", "kind": "ic", "n": 1024},
        # a few binaries: each one's serial chain of steps is the time
        {"name": "trajectory_16", "kind": "trajectory", "n": 16, "rtol": 1e-10},
        # more binaries than the chip holds at once
        {"name": "trajectory_4096", "kind": "trajectory", "n": 4096, "rtol": 1e-10},
        # long templates: 5k to 60k knots each
        {"name": "splines_512", "kind": "splines", "n": 512, "kmin": 5000, "kmax": 60000},
        # the reference's five modes on 256 s at 4096 Hz
        {"name": "modes_512", "kind": "modes", "n": 512, "nm": 5, "N": 1 << 20, "rate": 4096},
        # inspiral-merger-ringdown templates of five modes on 64 s at 16384 Hz
        {"name": "imr_512", "kind": "imr", "n": 512, "nm": 5, "N": 1 << 20, "rate": 16384},
        # log L of a proposal batch of 1024 templates against 256 s of data
        {"name": "likelihood_1024", "kind": "likelihood", "n": 1024, "N": 1 << 20, "rate": 4096},
        # the same number the reference's way: every template transformed at full length
        {"name": "direct_256", "kind": "direct", "n": 256, "N": 1 << 20, "rate": 4096},
        # what an injection study writes out: three interferometers' signals
        {"name": "detector_256", "kind": "detector", "n": 256, "N": 1 << 20, "rate": 4096, "nifo": 3},
        # the reference's template path on a small batch and a short segment, as drop-ins
        {"name": "dropin_32", "kind": "dropin", "n": 32, "knots": 2048, "nm": 5, "N": 1 << 17, "rate": 4096, "nifo": 3},
        # the headline: 1024 fresh proposals, parameters to log L
        {"name": "pass_1024", "kind": "pass", "n": 1024, "N": 1 << 20, "rate": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "ic", "trajectory", "splines", "modes", "imr", "likelihood", "direct", "detector", "dropin", "pass"))
    c = {"kind": kind}
    if kind == "step":
        c["n"] = _log(rng, 1, 2048)
    elif kind == "ic":
        c["n"] = _log(rng, 1, 2048)
    elif kind == "trajectory":
        c["n"] = _log(rng, 1, 3500)
        c["rtol"] = rng.choice((1e-10, 1e-9, 1e-8))
    elif kind == "splines":
        c["n"] = _log(rng, 2, 512)
        c["kmin"] = _log(rng, 5, 5000)
        c["kmax"] = min(60000, c["kmin"] * rng.randint(2, 12))
    elif kind in ("modes", "imr"):
        c["n"] = _log(rng, 2, 512)
        c["nm"] = rng.randint(1, 8 if kind == "modes" else 5)
        c["N"] = _log(rng, 1 << 12, 1 << 20)
        c["rate"] = rng.choice((2048, 4096) if kind == "modes" else (4096, 16384))
    elif kind in ("likelihood", "pass"):
        c["n"] = _log(rng, 2, 1024)
        c["N"] = 1 << rng.randint(14, 20)
        c["rate"] = rng.choice((2048, 4096))
    elif kind in ("direct", "detector"):
        c["n"] = _log(rng, 1, 256)
        c["N"] = 1 << rng.randint(11, 20) if rng.random() < 0.7 else 2 * _log(rng, 1000, 1 << 19)
        c["rate"] = rng.choice((2048, 4096))
        if kind == "detector":
            c["nifo"] = rng.randint(1, 5)
    else:
        c["n"] = _log(rng, 1, 64)
        c["knots"] = _log(rng, 20, 4096)
        c["nm"] = rng.randint(1, 5)
        c["N"] = 1 << rng.randint(10, 17) if rng.random() < 0.7 else 2 * _log(rng, 500, 1 << 16)
        c["rate"] = rng.choice((2048, 4096))
        c["nifo"] = rng.randint(1, 3)
    return c


# ------------------------------------------------------------------ inputs
def _dev(x):
    return torch.as_tensor(np.ascontiguousarray(x, dtype=np.float64), device="cuda")


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) + 1)


def _binaries(n, seed):
    return configs.uneven_batch(n=n, seed=seed)


def _trajectories(n, seed, max_step=4096):
    """A batch with its trajectories integrated: what every later stage starts from."""
    p = _binaries(n, seed)
    b = pipeline.EOBBatch.from_params(p["m1"], p["m2"], p["chi1"], p["chi2"], max_step=max_step)
    b.initial_conditions(p["r0"])
    b.integrate(rtol=1e-10, atol=1e-10, two_pass=True)
    return p, b


def _splined(n, seed):
    p, b = _trajectories(n, seed)
    b.hlm22_knots()
    b.coef = torch.zeros((n, b.max_step, 12), dtype=torch.float64, device="cuda")
    b.spline_scratch = torch.empty(int(pipeline.lib().eobhip_spline_scratch_doubles(n, b.max_step)), dtype=torch.float64, device="cuda")
    b.build_splines()
    return p, b


def _noise_curve(F, df):
    x = torch.arange(F, dtype=torch.float64, device="cuda") * df / F0
    w = x ** 4 / (1.0 + x ** 4 + x ** 6)
    return w   # 1 / S, 0 at f = 0


def _data(b, M, N, dt, seed):
    """Stationary noise with the analytic curve plus binary 0 at SNR 20; returns (data, amplitude)."""
    F, df = N // 2 + 1, 1.0 / (N * dt)
    w = _noise_curve(F, df)
    g = _gen(seed)
    noise = torch.randn(2, F, dtype=torch.float64, device="cuda", generator=g)
    sig = torch.where(w > 0, 1.0 / torch.sqrt(w.clamp(min=1e-300)), 0.0) / math.sqrt(8 * df)
    d = torch.complex(noise[0] * sig, noise[1] * sig)
    h0 = torch.fft.rfft(_hplus_exact(b, M, dt, N, 0, 1, 1.0)[0].real[0])
    rho = torch.sqrt(4 * df * (h0.abs() ** 2 * w).sum())
    amp = float(20.0 / rho)
    return (d + h0 * amp).contiguous(), amp


def _sky(n, nifo, seed):
    rng = np.random.default_rng(seed + 23)
    D, V = [], []
    for _ in range(nifo):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        D.append(0.5 * (np.outer(q[:, 0], q[:, 0]) - np.outer(q[:, 1], q[:, 1])))
        V.append(q[:, 2] * 6.4e6)
    ang = dict(ra=rng.uniform(0, 2 * np.pi, n), dec=np.arcsin(rng.uniform(-1, 1, n)), gmst=rng.uniform(0, 2 * np.pi, n),
               psi=rng.uniform(0, np.pi, n))
    return {k: _dev(v) for k, v in ang.items()}, _dev(np.array(D)), _dev(np.array(V))


def _chirps(n, kmin, kmax, N, dt, M, seed, amp=1e-21):
    """Knot times (units of M), phase and amplitude of n chirps with kmin .. kmax knots
    (``configs.chirp_modes``' distributions, made on the device)."""
    g = _gen(seed)
    K = torch.randint(kmin, kmax + 1, (n,), generator=g, device="cuda")
    L = kmax
    u = (1.0 - 2e-6) * torch.rand(n, L, dtype=torch.float64, device="cuda", generator=g)
    col = torch.arange(L, device="cuda")
    # rows end at their own length: the rest is pushed past 1 before the sort
    u = torch.where(col[None, :] < K[:, None], u, 2.0).sort(dim=1).values
    u[:, 0] = 0.0
    u.scatter_(1, (K - 1)[:, None], 1.0 - 1e-6)
    valid = col[None, :] < K[:, None]
    u = torch.where(valid, u, 0.0)
    T = N * dt / (M * MTSUN) * (0.05 + 0.85 * torch.rand(n, 1, dtype=torch.float64, device="cuda", generator=g))
    t = T * (1.0 - (1.0 - u) ** 0.375)
    x = 1.0 - t / T
    phi = math.pi * 20.0 * M * MTSUN * T * 1.6 * (1.0 - x ** 0.625)
    z = torch.zeros((), dtype=torch.float64, device="cuda")
    return K, torch.where(valid, t, z), torch.where(valid, phi, z), torch.where(valid, amp * x ** -0.25, z)


_handle = {}   # the streamed pass of the newest batch shape, kept as a sampler's program keeps it


def _streamed(n, N, rate):
    key = (n, N, rate)
    if key not in _handle:
        _handle.clear()
        p, b = _splined(n, 2)
        M = p["m1"] + p["m2"]
        d, amp = _data(b, M, N, 1.0 / rate, 7)
        lik = pipeline.SupportLikelihood(d, N, rate / N, f0=F0)
        sp = pipeline.StreamedPass(p["m1"], p["m2"], p["chi1"], p["chi2"], p["r0"], lik, M, 1.0 / rate, amp=np.full(n, amp))
        _handle[key] = (sp, amp)
    return _handle[key]


def prepare(case, seed):
    k, n = case["kind"], case["n"]
    s = dict(case)
    if k in ("step", "ic"):
        p = _binaries(n, seed)
        om = 20.0 * math.pi * (p["m1"] + p["m2"]) * MTSUN if k == "ic" else None
        add = pipeline.make_additional_args(p["m1"], p["m2"], p["chi1"], p["chi2"], omega0=om)
        m1, m2, c1, c2 = add[:4]
        eta = m1 * m2 / (m1 + m2) ** 2
        cS, cA = 0.5 * (c1 + c2), 0.5 * (c1 - c2)
        ode = pyEOB.SEOBNRv5Class()
        s["pref"] = _dev(add[10:80].T)
        ode.update_information(_dev(m1), _dev(m2), _dev(eta), _dev((1 - 2 * eta) * cS + (m1 - m2) / (m1 + m2) * cA), _dev(cS), _dev(cA),
                               1, n, s["pref"])
        s["ode"], s["add0"] = ode, _dev(add).reshape(-1)
        if k == "ic":
            rg = om ** (-2.0 / 3)
            s["x0"] = _dev(np.array([rg, np.sqrt(rg)])).reshape(-1)
            s["bounds"] = _dev(np.array([np.full(n, -3e-2), np.zeros(n)])).reshape(-1)
            return s
        # states along a quasi-circular inspiral, steps of a fraction of a radian
        rng = np.random.default_rng(seed + 5)
        r = rng.uniform(8.0, 40.0, n)
        L = np.sqrt(r) * (1 + 1.5 / r + 27.0 / 8 / r ** 2)
        y = np.array([r, rng.uniform(0, 100.0, n), -64.0 / 5 * eta / r ** 3, L])
        s["y"], s["h0"], s["x"] = _dev(y).reshape(-1), _dev(rng.uniform(0.2, 0.9, n) * r ** 1.5), _dev(rng.uniform(0, 1e4, n))
        s["idx"] = torch.arange(n, dtype=torch.int32, device="cuda")
        buf = lambda m: torch.zeros(m, dtype=torch.float64, device="cuda")  # noqa: E731
        s.update(k=[buf(4 * n) for _ in range(10)], arg=buf(4 * n), ak=buf(4 * n), new=buf(4 * n), xc=buf(n), err=buf(n))
        return s
    if k == "trajectory":
        p = _binaries(n, seed)
        s["b"] = pipeline.EOBBatch.from_params(p["m1"], p["m2"], p["chi1"], p["chi2"])
        s["par"] = [_dev(p[q]) for q in ("m1", "m2", "chi1", "chi2", "r0")]
        return s
    if k == "splines":
        K, t, phi, a = _chirps(n, case["kmin"], case["kmax"], 1 << 20, 1.0 / 4096, 30.0, seed)
        L = int(t.shape[1])
        b = pipeline.EOBBatch.from_params(np.full(n, 0.6), np.full(n, 0.4), np.zeros(n), np.zeros(n), max_step=L)
        b.dense[:, :, 0] = t
        b.num_steps.copy_(K.to(torch.int32))
        b.knots = torch.stack([phi, a, 0.3 * a * torch.sin(phi / 40.0)], dim=2).contiguous()
        b.coef = torch.zeros((n, L, 12), dtype=torch.float64, device="cuda")
        b.spline_scratch = torch.empty(int(pipeline.lib().eobhip_spline_scratch_doubles(n, L)), dtype=torch.float64, device="cuda")
        s["b"] = b
        return s
    if k in ("modes", "imr"):
        p, b = _trajectories(n, seed)
        s["b"], s["M"], s["modes"] = b, p["m1"] + p["m2"], MODES[:case["nm"]]
        s["knots"] = torch.zeros((n, b.max_step, 2 * case["nm"] + 1), dtype=torch.float64, device="cuda")
        return s
    if k == "pass":
        sp, amp = _streamed(n, case["N"], case["rate"])
        p = _binaries(n, seed)
        s["sp"] = sp
        s["par"] = _dev(np.stack([p["m1"], p["m2"], p["chi1"], p["chi2"], p["r0"], p["m1"] + p["m2"], np.full(n, amp)]))
        return s
    if k in ("likelihood", "direct", "detector"):
        N, dt = case["N"], 1.0 / case["rate"]
        p, b = _splined(n, seed)
        s["b"], s["M"] = b, p["m1"] + p["m2"]
        if k == "detector":
            s["sky"], s["D"], s["V"] = _sky(n, case["nifo"], seed)
            return s
        d, amp = _data(b, s["M"], N, dt, seed)
        s["data"], s["amp"] = d, np.full(n, amp)
        if k == "likelihood":
            s["lik"] = pipeline.SupportLikelihood(d, N, 1.0 / (N * dt), f0=F0)
        return s
    # dropin: knots of nm modes in the reference's layouts, times in seconds
    N, dt, nk, nm, nifo = case["N"], 1.0 / case["rate"], case["knots"], case["nm"], case["nifo"]
    S = 2 * nm + 1
    K, t, phi, a = _chirps(n, max(4, nk // 2), nk, N, dt, 30.0, seed, amp=1.0)
    L = int(t.shape[1])
    sec = t * (30.0 * MTSUN)
    valid = torch.arange(L, device="cuda")[None, :] < K[:, None]
    y = torch.zeros((n, S, L), dtype=torch.float64, device="cuda")
    for q in range(nm):
        y[:, q] = a * torch.cos(0.1 * q + 0.02 * phi) / (1 + q)
        y[:, nm + q] = a * torch.sin(0.1 * q + 0.02 * phi) / (1 + q)
    y[:, 2 * nm] = phi
    y = torch.where(valid[:, None, :], y, 0.0).contiguous()
    s["y"], s["ts"] = y, torch.where(valid, sec, float("inf")).contiguous()
    s["t_len"] = sec.T.contiguous()                              # [L][n]
    s["y_len"] = y.permute(2, 1, 0).reshape(L, S * n).contiguous()   # [L][S n]
    s["K"] = K.to(torch.int32)
    s["time"] = torch.arange(N, dtype=torch.float64, device="cuda") * dt
    last = sec.gather(1, (K - 1)[:, None])[:, 0]
    s["count"] = torch.searchsorted(s["time"], last, right=True).clamp(max=N).to(torch.int32)
    ind = torch.searchsorted(s["ts"], s["time"].expand(n, N).contiguous(), right=True) - 1
    s["inds"] = torch.minimum(ind.clamp(min=0), (K - 2)[:, None]).to(torch.int32).contiguous()
    s["ls"] = torch.tensor([m[0] for m in MODES[:nm]], dtype=torch.int32, device="cuda")
    s["ms"] = torch.tensor([m[1] for m in MODES[:nm]], dtype=torch.int32, device="cuda")
    F, df = N // 2 + 1, 1.0 / (N * dt)
    g = _gen(seed + 1)
    w = _noise_curve(F, df)
    s["psd"] = (1.0 / w.clamp(min=1e-12)).expand(nifo, F).contiguous()
    nz = torch.randn(2, nifo, F, dtype=torch.float64, device="cuda", generator=g)
    s["data"] = torch.complex(nz[0], nz[1]) * torch.sqrt(s["psd"])
    rnd = torch.rand(3, nifo * n, dtype=torch.float64, device="cuda", generator=g)
    s["Fp"], s["Fc"], s["shift"] = 2 * rnd[0] - 1, 2 * rnd[1] - 1, 0.02 * (2 * rnd[2] - 1)
    z = lambda *q, dtype=torch.float64: torch.zeros(q, dtype=dtype, device="cuda")  # noqa: E731
    s.update(L=L, B=z(L, S * n), c1=z(L, S * n), c2=z(L, S * n), c3=z(L, S * n), out=z(n, N, dtype=torch.complex128),
             sums=z((F + 1023) // 1024 * n * nifo, dtype=torch.complex128), df=df)
    return s


# --------------------------------------------------------------------- run
def run(s):
    k, n = s["kind"], s["n"]
    if k == "step":
        h, x, add = s["h0"].clone(), s["x"].clone(), s["add0"]
        err_old = torch.full((n,), 1e-4, dtype=torch.float64, device="cuda")
        flag, rej = torch.zeros(n, dtype=torch.bool, device="cuda"), torch.zeros(n, dtype=torch.bool, device="cuda")
        ks = s["k"]
        pydopr853.dormandPrinceSteps(x, s["xc"], s["y"], h, s["arg"], add, *ks, s["ak"], 4, n, 80, s["ode"], s["idx"])
        pydopr853.error(s["err"], s["y"], s["new"], h, ks[0], ks[1], ks[2], ks[5], ks[6], ks[7], ks[8], ks[9], n, 4)
        pydopr853.controllerSuccess(flag, s["err"], err_old, rej, h, x, n, 4)
        return {"new": s["new"], "err": s["err"], "h": h, "err_old": err_old, "flag": flag, "rejected": rej, "k": list(ks),
                "x_stage": s["xc"]}
    if k == "ic":
        add = s["add0"].clone()
        xo = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
        args = torch.zeros(4 * n, dtype=torch.float64, device="cuda")
        pyEOB.root_find_all(xo, s["x0"], args, add, 1000, 1e-12, n, 2, 4, 80)
        args.view(4, n)[0] = xo[:n]
        args.view(4, n)[3] = xo[n:]
        pr = torch.zeros(n, dtype=torch.float64, device="cuda")
        s["ode"].root_find_scalar_all(pr, s["bounds"], args, add, 1000, 1e-12, n, 4, 80)
        return {"x": xo, "pr": pr}
    if k == "trajectory":
        b = s["b"]
        b.set_params(*s["par"][:4])
        b.initial_conditions(s["par"][4])
        b.integrate(rtol=s["rtol"], atol=s["rtol"], two_pass=True)
        return {"dense": b.dense, "num_steps": b.num_steps, "stop": b.stop_info, "pass1": b.pass1_steps, "attempts": b.attempts}
    if k == "splines":
        return s["b"].build_splines()
    if k in ("modes", "imr"):
        b = s["b"]
        b.hlm_modes_knots(s["modes"], out=s["knots"])
        b.build_mode_splines()
        f = b.resample_modes if k == "modes" else b.imr_template
        hp, hc = f(s["M"], 1.0 / s["rate"], s["N"])
        return {"knots": s["knots"], "hp": hp, "hc": hc}
    if k == "likelihood":
        terms = torch.empty((n, 2), dtype=torch.float64, device="cuda")
        logl = s["lik"](s["b"], s["M"], 1.0 / s["rate"], amp=s["amp"], terms=terms)
        return {"logl": logl, "terms": terms}
    if k == "direct":
        b = s["b"]
        b.hlm22_knots(out=b.knots)
        b.build_splines()
        hp = b.resample_hplus(s["M"], 1.0 / s["rate"], s["N"], amp=s["amp"])
        ht = pipeline.rfft_batched(hp)
        return {"coef": b.coef, "hp": hp, "ht": ht, "logl": pipeline.fd_likelihood(ht, s["data"], s["rate"] / s["N"], f0=F0)}
    if k == "detector":
        hp, hc = detector.resample_hpc(s["b"], s["M"], 1.0 / s["rate"], s["N"])
        hpf, hcf = pipeline.rfft_batched(hp), pipeline.rfft_batched(hc)
        q = s["sky"]
        Fp, Fc, ts = detector.get_detector_information(q["ra"], q["dec"], q["gmst"], q["psi"], s["D"], s["V"])
        return {"Fp": Fp, "Fc": Fc, "shift": ts,
                "signal": detector.detector_signal(hpf, hcf, Fp, Fc, ts, s["rate"] / s["N"], k_min=(20 * s["N"]) // s["rate"])}
    if k == "dropin":
        L, nm, N = s["L"], s["nm"], s["N"]
        S = 2 * nm + 1
        pytdinterp.interpolate_TD_wrap(s["t_len"], s["y_len"], s["B"], s["c1"], s["c2"], s["c3"], s["K"], n, S)
        c = [s[q].view(L, S, n).permute(2, 1, 0).contiguous() for q in ("c1", "c2", "c3")]
        pytdinterp.TDInterp_wrap2(s["out"], s["time"], s["ts"], s["y"], *c, L, s["K"], N, n, nm, s["ls"], s["ms"], s["inds"], s["count"], N,
                                  legacy_stride=False)
        hp, hc = (pipeline.rfft_batched(q.contiguous()) for q in (s["out"].real, s["out"].imag))
        pytdinterp.all_in_one_likelihood(s["sums"], hp, hc, s["data"], s["psd"], s["Fp"], s["Fc"], s["shift"], s["df"], n, s["nifo"], N // 2 + 1)
        return {"template": s["out"], "sums": s["sums"]}
    s["sp"].set_params_device(s["par"])
    s["sp"].run()
    return s["sp"].out.clone()


# -------------------------------------------------------------------- work
def work(case):
    """What each input read once and each output written once moves, and the FP64
    operations of the arithmetic the outputs are defined by."""
    k, n, N = case["kind"], case["n"], case.get("N", 0)
    F = N // 2 + 1
    fft = 2.5 * N * math.log2(max(N, 2))      # a real transform of N samples
    if k == "step":
        return {"bytes": n * 8.0 * (80 + 35 * 32 + 4 * 14), "flops": n * float(STEP_FLOPS)}
    if k == "ic":
        return {"bytes": n * 8.0 * (80 + 35 * 32 + 8), "flops": n * (18 * 1600.0 + 8 * (RHS_FLOPS + 2000.0))}
    if k == "trajectory":
        return {"bytes": n * 40.0 * KNOTS, "flops": n * float(ATTEMPTS) * STEP_FLOPS}
    if k == "splines":
        m = n * 0.5 * (case["kmin"] + case["kmax"])
        return {"bytes": m * 128.0, "flops": m * 3 * 30.0}
    if k in ("modes", "imr"):
        nm = case["nm"]
        return {"bytes": n * (16.0 * N + KNOTS * 8.0 * (5 + 5 * (2 * nm + 1))), "flops": n * (0.25 * N * (40 + 30 * nm) + KNOTS * 400.0 * nm)}
    if k == "likelihood":
        # coefficients and the data's two weights read, log L written; supports are a tenth of the segment
        return {"bytes": n * 96.0 * KNOTS + 16.0 * N, "flops": n * 0.1 * (2.5 * 2 * N * math.log2(N) + 60.0 * N)}
    if k == "direct":
        return {"bytes": n * (8.0 * N + 16.0 * F + KNOTS * 136.0) + 16.0 * F, "flops": n * (fft + 10.0 * F)}
    if k == "detector":
        return {"bytes": n * (16.0 * F * case["nifo"] + KNOTS * 136.0), "flops": n * (2 * fft + 14.0 * F * case["nifo"])}
    if k == "dropin":
        S = 2 * case["nm"] + 1
        return {"bytes": n * (case["knots"] * 8.0 * (1 + 4 * S) + 16.0 * N + 4.0 * N) + 24.0 * F * case["nifo"],
                "flops": n * (2 * fft + N * (6.0 * S + 30) + 20.0 * F * case["nifo"])}
    return {"bytes": n * 8.0 * 8 + 16.0 * N, "flops": n * float(ATTEMPTS) * STEP_FLOPS}


# ------------------------------------------------------------------- exact
def _hplus_exact(b, M, dt, N, lo, hi, amp):
    """(h [hi-lo][N] complex, samples [hi-lo]) of binaries lo .. hi-1 from the batch's
    (2,2) spline coefficients: amp S(t) e^{-2 i phi(t)} on t_0 + j dt, zero past the last knot."""
    ns = b.num_steps[lo:hi].to(torch.int64)
    dT = dt / (_dev(M[lo:hi]) * MTSUN)
    t = b.dense[lo:hi, :, 0]
    L = t.shape[1]
    valid = torch.arange(L, device="cuda")[None, :] < ns[:, None]
    ts = torch.where(valid, t, float("inf")).contiguous()
    t0 = t[:, :1]
    tl = t.gather(1, (ns - 1).clamp(min=0)[:, None])
    nb = torch.where(ns[:, None] >= 2, torch.floor((tl - t0) / dT[:, None]) + 1, 0.0).clamp(max=N)
    j = torch.arange(N, dtype=torch.float64, device="cuda")[None, :]
    tj = t0 + j * dT[:, None]
    ind = (torch.searchsorted(ts, tj, right=True) - 1).clamp(min=0)
    ind = torch.minimum(ind, (ns - 1).clamp(min=0)[:, None])
    x = tj - torch.where(valid, t, 0.0).gather(1, ind)
    def series(q):
        c = [b.coef[lo:hi, :, 4 * q + i].gather(1, ind) for i in range(4)]
        return c[0] + x * (c[1] + x * (c[2] + x * c[3]))
    ph = series(0)
    h = amp * torch.polar(torch.ones_like(ph), -2 * ph) * torch.complex(series(1), series(2))
    return torch.where(j < nb, h, 0.0), nb[:, 0].to(torch.int64)


def _spline_exact(t, y, K):
    """Not-a-knot coefficients c1, c2, c3 of y [R][L] over t [R][L], K [R] knots (>= 4; zero
    from row K - 1 on), by cyclic reduction of the slope system on all rows at once."""
    R, L = y.shape
    i = torch.arange(L, device=t.device)[None, :]
    last = (K - 1)[:, None]
    dx = torch.ones_like(t)
    dx[:, :-1] = t[:, 1:] - t[:, :-1]
    dx = torch.where(i < last, dx, 1.0)
    m = torch.zeros_like(y)
    m[:, :-1] = (y[:, 1:] - y[:, :-1]) / dx[:, :-1]
    m = torch.where(i < last, m, 0.0)
    at = lambda v, k: v.gather(1, k.expand(R, 1))  # noqa: E731
    p = lambda v: torch.cat([v[:, :1], v[:, :-1]], 1)  # noqa: E731  (the row below)
    a, d, c = dx.clone(), 2 * (p(dx) + dx), p(dx).clone()
    r = 3.0 * (dx * p(m) + p(dx) * m)
    # the end rows, solved into their neighbours: row 0: dx1 s0 + (dx0 + dx1) s1 = b0; the last likewise
    dx0, dx1, m0, m1 = dx[:, :1], dx[:, 1:2], m[:, :1], m[:, 1:2]
    b0 = ((dx0 + 2 * (dx0 + dx1)) * dx1 * m0 + dx0 ** 2 * m1) / (dx0 + dx1)
    ea, eb, ma, mb = at(dx, last - 2), at(dx, last - 1), at(m, last - 2), at(m, last - 1)
    bl = (eb ** 2 * ma + (2 * (ea + eb) + eb) * ea * mb) / (ea + eb)
    one = i == 1
    d, r, a = torch.where(one, d - (dx0 + dx1), d), torch.where(one, r - b0, r), torch.where(one, 0.0, a)
    pen = i == last - 1   # the row before the last: subtract the last row
    d, r, c = torch.where(pen, d - (ea + eb), d), torch.where(pen, r - bl, r), torch.where(pen, 0.0, c)
    inside = (i >= 1) & (i <= last - 1)
    a, c, r, d = (torch.where(inside, v, f) for v, f in ((a, 0.0), (c, 0.0), (r, 0.0), (d, 1.0)))
    k = 1
    def sh(v, s, fill):
        o = torch.full_like(v, fill)
        if s > 0:
            o[:, s:] = v[:, :-s]
        else:
            o[:, :s] = v[:, -s:]
        return o
    while k < L:
        al, ga = -a / sh(d, k, 1.0), -c / sh(d, -k, 1.0)
        d = d + al * sh(c, k, 0.0) + ga * sh(a, -k, 0.0)
        r = r + al * sh(r, k, 0.0) + ga * sh(r, -k, 0.0)
        a, c = al * sh(a, k, 0.0), ga * sh(c, -k, 0.0)
        k *= 2
    sl = r / d
    s0 = (b0 - (dx0 + dx1) * sl[:, 1:2]) / dx1
    sn = (bl - (ea + eb) * at(sl, last - 1)) / ea
    sl = torch.where(i == 0, s0, torch.where(i == last, sn, sl))
    nx = torch.cat([sl[:, 1:], sl[:, -1:]], 1)
    tt = (sl + nx - 2 * m) / dx
    keep = i < last
    return torch.where(keep, sl, 0.0), torch.where(keep, (m - sl) / dx - tt, 0.0), torch.where(keep, tt / dx, 0.0)


def exact(case, seed):
    k, n = case["kind"], case["n"]
    if k == "splines":
        if case["kmin"] < 4:
            return None
        b = prepare(case, seed)["b"]
        K = b.num_steps.to(torch.int64)
        out = torch.zeros_like(b.coef)
        L = b.max_step
        valid = torch.arange(L, device="cuda")[None, :] < K[:, None]
        for lo in range(0, n, 64):
            t, kk, v = b.dense[lo:lo + 64, :, 0], K[lo:lo + 64], valid[lo:lo + 64]
            for q in range(3):
                y = b.knots[lo:lo + 64, :, q]
                out[lo:lo + 64, :, 4 * q] = torch.where(v, y, 0.0)
                for e, c in enumerate(_spline_exact(t, y, kk)):
                    out[lo:lo + 64, :, 4 * q + 1 + e] = c
        return out
    if k in ("likelihood", "direct", "detector"):
        s = prepare(case, seed)
        b, N, dt = s["b"], case["N"], 1.0 / case["rate"]
        F, df = N // 2 + 1, 1.0 / (N * dt)
        step = max(1, (1 << 24) // N)
        w = _noise_curve(F, df)
        if k == "likelihood":
            d, logl, terms = s["data"], [], []
            for lo in range(0, n, step):
                hi = min(n, lo + step)
                ht = torch.fft.rfft(_hplus_exact(b, s["M"], dt, N, lo, hi, s["amp"][0])[0].real)
                logl.append(-2 * df * ((d - ht).abs() ** 2 * w).sum(1))
                terms.append(torch.stack([((d.conj() * ht).real * w).sum(1), (ht.abs() ** 2 * w).sum(1)], 1))
            return {"logl": torch.cat(logl), "terms": torch.cat(terms)}
        if k == "direct":
            d, hp, ht, logl = s["data"], [], [], []
            for lo in range(0, n, step):
                hi = min(n, lo + step)
                hp.append(_hplus_exact(b, s["M"], dt, N, lo, hi, s["amp"][0])[0].real)
                ht.append(torch.fft.rfft(hp[-1]))
                logl.append(-2 * df * ((d - ht[-1]).abs() ** 2 * w).sum(1))
            return {"coef": None, "hp": torch.cat(hp), "ht": torch.cat(ht), "logl": torch.cat(logl)}
        q, nifo = s["sky"], case["nifo"]
        phi, th, ps = q["ra"] - q["gmst"], 0.5 * math.pi - q["dec"], q["psi"]
        u = torch.stack([phi.cos() * th.cos(), th.cos() * phi.sin(), -th.sin()])
        v = torch.stack([-phi.sin(), phi.cos(), torch.zeros_like(phi)])
        m, e = -u * ps.sin() - v * ps.cos(), -u * ps.cos() + v * ps.sin()
        D, V = s["D"].reshape(nifo, 3, 3), s["V"]
        dot = lambda x, y: torch.stack([(Di @ y * x).sum(0) for Di in D])  # noqa: E731
        Fp, Fc = dot(m, m) - dot(e, e), dot(m, e) + dot(e, m)
        om = torch.stack([th.sin() * phi.cos(), th.sin() * phi.sin(), th.cos()])
        ts = V @ om / 299792458.0
        f = torch.arange(F, dtype=torch.float64, device="cuda") * df
        keep = torch.arange(F, device="cuda") >= (20 * N) // case["rate"]
        sig = torch.empty((n, nifo, F), dtype=torch.complex128, device="cuda")
        for lo in range(0, n, step):
            hi = min(n, lo + step)
            h = _hplus_exact(b, s["M"], dt, N, lo, hi, 1.0)[0]
            p, c = torch.fft.rfft(h.real), torch.fft.rfft(h.imag)
            for i in range(nifo):
                z = Fp[i, lo:hi, None] * p + Fc[i, lo:hi, None] * c
                ph = -2 * math.pi * (f[None, :] * ts[i, lo:hi, None])
                sig[lo:hi, i] = torch.where(keep, z * torch.polar(torch.ones_like(ph), ph), 0.0)
        return {"Fp": Fp, "Fc": Fc, "shift": ts, "signal": sig}
    if k == "dropin":
        s = prepare(case, seed)
        L, nm, N, nifo, F, df = s["L"], s["nm"], s["N"], s["nifo"], s["N"] // 2 + 1, s["df"]
        K = s["K"].to(torch.int64)
        t = torch.where(torch.isfinite(s["ts"]), s["ts"], 0.0)
        ind = s["inds"].to(torch.int64)
        x = s["time"][None, :] - t.gather(1, ind)
        def series(q):
            y = s["y"][:, q]
            c = _spline_exact(t, y, K)
            return y.gather(1, ind) + x * (c[0].gather(1, ind) + x * (c[1].gather(1, ind) + x * c[2].gather(1, ind)))
        phi = series(2 * nm)
        h = torch.zeros((n, N), dtype=torch.complex128, device="cuda")
        for q in range(nm):
            ph = -float(s["ms"][q]) * phi
            h += torch.complex(series(q), series(nm + q)) * torch.polar(torch.ones_like(ph), ph)
        h = torch.where(torch.arange(N, device="cuda")[None, :] < s["count"][:, None], h, 0.0)
        p, c = torch.fft.rfft(h.real), torch.fft.rfft(h.imag)
        f = torch.arange(F, dtype=torch.float64, device="cuda") * df
        nblk = (F + 1023) // 1024
        sums = torch.zeros((nblk, n, nifo), dtype=torch.complex128, device="cuda")
        Fp, Fc, sh = (s[q].view(nifo, n) for q in ("Fp", "Fc", "shift"))
        for i in range(nifo):
            ph = -2 * math.pi * (f[None, :] * sh[i][:, None])
            z = (Fp[i][:, None] * p + Fc[i][:, None] * c) * torch.polar(torch.ones_like(ph), ph)
            v = torch.zeros((n, nblk * 1024), dtype=torch.float64, device="cuda")
            v[:, :F] = (s["data"][i] - z).abs() ** 2 / s["psd"][i]
            sums[:, :, i] = v.view(n, nblk, 1024).sum(2).T
        return {"template": h, "sums": sums.reshape(-1)}
    return None
