"""The workloads that this framework is timed on: what a user has it do, through its public entry points.

Seven kinds of work:

    fit      a whole fit from host arrays (``engine.run_fits``): upload, random start, burn-in, sampling with every
             sample recorded, download.
    sample   iterations of a resident session (``engine.Session``) and the download of the chains' state.
    batch    the same for a session of many uneven fits.
    quad     the same for a session of many quadratic systems.
    grad     chi^2 and its gradient for a batch of parameter rows (``adjoint.chi2`` and its backward).
    normal   chi^2 and the Gauss-Newton normal equations of parameter rows (``EhtData.gn_system``).
    chi2     model data and chi^2 of host parameter rows (``mcmc_interf.calcmodchi2``).

Sizes are those of the benchmark (bench.py), the examples and the tests.
"""
import math
import os

import numpy as np
import torch

from cuda_mcmc_amd import adjoint, mcmc_interf, quadsys, synthdata
from cuda_mcmc_amd.engine import Fit, Session, run_fits

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FOREVER = 1 << 30   # iterations of a session that never reaches its end

# the 13-parameter prior box: Zsp Re rq ecc fade gr gax aq gq alpha beta eta th
PI = math.pi
P13_MIN = np.array([0.5, 20., 0.3, 0.0, 0.0, 0.0, 1.6, 0.5, 0.0, -PI, -PI, -PI, -PI], np.float32)
P13_MAX = np.array([3.0, 30., 0.9, 0.5, 1.0, 1.0, 7.5, 1.0, 0.5, PI, PI, PI, PI], np.float32)
P13_DESCR = np.array([1] * 9 + [2] * 4, np.int32)

# flops of one visibility, one closure phase and one chi^2 evaluation (bench.py)
F_VIS, F_CPH, F_CHAIN = 170.0, 15.0, 40.0


def listed():
    return [
        # the two-parameter example in its stated size: one datum, so launches and latency are all there is
        dict(name="rosenbrock_fit", kind="fit", model="rosenbrock", nbeta=32, nseq=64, nburn=2000, niter=5000),
        # the size of the reference's observation fit: 323 visibilities, 32 x 16 chains, 400 + 1000 iterations
        dict(name="observation_fit", kind="fit", model="sgra9", nvis=323, ncph=319, nsta=8, cpext=0, nbeta=32, nseq=16,
             nburn=400, niter=1000),
        # the 13-parameter model in the driver's default run shape, closures from their own (u, v) points
        dict(name="fit_13_parameters", kind="fit", model="sgra13", nvis=323, ncph=319, nsta=8, cpext=1, nbeta=32,
             nseq=14, nburn=300, niter=500),
        # the same observation through a user's own model.cuh (one model() call per datum)
        dict(name="user_model_fit", kind="fit", model="user", nvis=323, ncph=319, nsta=8, cpext=0, nbeta=32, nseq=16,
             nburn=10, niter=10),
        # the benchmark's plain fit, after burn-in: 2000 visibilities + 600 closures, 4096 chains
        dict(name="plain_sampling", kind="sample", nvis=2000, ncph=600, nsta=8, nbeta=32, nseq=128, nburn=300,
             iters=500),
        # uneven fits (500 - 20000 visibilities, ladders of 16 - 48 rungs) in one session, in burn-in
        dict(name="batch_burn_in", kind="batch", fits=12, layout=1, iters=40),
        # quadratic systems: the whole burn-in stage, and half of the sampling stage
        dict(name="quad_burn_in", kind="quad", nsys=512, n=8, nbeta=16, nseq=32, burn=True, iters=3000),
        dict(name="quad_sampling", kind="quad", nsys=512, n=8, nbeta=16, nseq=32, burn=False, iters=5000),
        # gradients at many points of a large observation, and at the best chains of a plain fit
        dict(name="gradient_4096_points", kind="grad", points=4096, nvis=20000, ncph=6000, nsta=8, near=False),
        dict(name="gradient_32_points", kind="grad", points=32, nvis=2000, ncph=600, nsta=8, near=True),
        # one Gauss-Newton / Laplace step of the best chains of a plain fit
        dict(name="normal_equations", kind="normal", points=16, nvis=2000, ncph=600, nsta=8),
        # model data and chi^2 of one state of the observation fit, host arrays in and out
        dict(name="model_and_chi2", kind="chi2", imodel=1, nvis=323, ncph=319, nsta=8, nbeta=32, nseq=16),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _max_closures(nvis, nsta):
    per_time, tri = nsta * (nsta - 1) // 2, nsta * (nsta - 1) * (nsta - 2) // 6
    return int(nvis / per_time * tri * 0.6)


def _observation(rng, nvis):
    nsta = rng.randint(5, 10)
    return dict(nvis=nvis, ncph=min(int(nvis * rng.choice([0.0, 0.3, 0.3, 0.95])), _max_closures(nvis, nsta)), nsta=nsta)


def draw(rng):
    kind = rng.choice(["small", "fit", "user", "sample", "batch", "quad", "grad", "normal", "chi2"])
    if kind == "small":
        return dict(kind="fit", model=rng.choice(["rosenbrock", "solvsys"]), nbeta=rng.randint(8, 48),
                    nseq=_logint(rng, 8, 128), nburn=rng.randint(200, 2000), niter=rng.randint(500, 3000))
    if kind == "fit":
        return dict(kind="fit", model=rng.choice(["sgra9", "sgra13"]), cpext=rng.choice([0, 0, 1]),
                    nbeta=rng.randint(8, 48), nseq=_logint(rng, 8, 64), nburn=rng.randint(100, 400),
                    niter=rng.randint(100, 500), **_observation(rng, _logint(rng, 100, 2000)))
    if kind == "user":
        return dict(kind="fit", model="user", cpext=0, nbeta=rng.randint(8, 48), nseq=_logint(rng, 4, 32),
                    nburn=rng.randint(2, 6), niter=rng.randint(2, 6), **_observation(rng, _logint(rng, 60, 500)))
    if kind == "sample":
        return dict(kind="sample", nbeta=rng.randint(16, 48), nseq=_logint(rng, 16, 128), nburn=rng.randint(50, 300),
                    iters=rng.randint(50, 200), **_observation(rng, _logint(rng, 500, 4000)))
    if kind == "batch":
        return dict(kind="batch", fits=rng.randint(3, 10), layout=rng.randint(2, 1 << 20), iters=rng.randint(10, 30))
    if kind == "quad":
        return dict(kind="quad", nsys=_logint(rng, 8, 400), n=rng.choice([2, 4, 8, 8]), nbeta=rng.randint(6, 32),
                    nseq=rng.randint(16, 48), burn=rng.random() < 0.5, iters=rng.randint(500, 3000))
    if kind == "grad":
        points = _logint(rng, 1, 2000)
        return dict(kind="grad", points=points, near=rng.random() < 0.5,
                    **_observation(rng, _logint(rng, 300, min(20000, 4000000 // points))))
    if kind == "normal":
        return dict(kind="normal", points=_logint(rng, 1, 300), **_observation(rng, _logint(rng, 300, 4000)))
    return dict(kind="chi2", imodel=rng.choice([1, 2]), nbeta=rng.randint(8, 48), nseq=_logint(rng, 4, 64),
                **_observation(rng, _logint(rng, 100, 2000)))


# ---------------------------------------------------------------------------------------------------- preparation

def _dataset(nvis, ncph, nsta, seed, cpext=0):
    d = synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, nsta=nsta, seed=seed)
    if cpext and ncph:   # the closures' own (u1, v1, u2, v2) behind the visibilities
        uv = d["coor"].reshape(-1, 2)
        ext = np.concatenate([uv[d["cpix"][:, 0]], uv[d["cpix"][:, 1]]], axis=1)
        d = dict(d, coor=np.concatenate([d["coor"], ext.ravel()]).astype(np.float32), cpext=1)
    return d


def _eht_fit(d, model, nbeta, nseq, seed, nburn, niter, **kw):
    if model == "sgra13":
        imodel, descr, lo, hi = 2, P13_DESCR, P13_MIN, P13_MAX
    else:
        imodel, descr, lo, hi = 1, synthdata.EHT_PDESCR, synthdata.EHT_PMIN, synthdata.EHT_PMAX
    idat = np.array([d["nvis"], nbeta * nseq * (d["nvis"] + d["ncph"]), d.get("cpext", 0)], np.int32)
    icoor = d["icoor"] if d["ncph"] else np.zeros(1, np.int32)
    return Fit(descr, lo, hi, d["coor"], d["dat"], d["std2r"], nbeta=nbeta, nseq=nseq, nburn=nburn, niter=niter,
               model="sgra13" if model == "sgra13" else "sgra9", imodel=imodel, icoor=icoor, idat=idat, npass=2,
               seed=seed, **kw)


def _layout(case):
    """The sizes of a batch's fits."""
    r = np.random.default_rng(case["layout"])
    out = []
    for _ in range(case["fits"]):
        nsta = int(r.integers(5, 11))
        nvis = int(np.exp(r.uniform(np.log(500), np.log(20000))))
        out.append(dict(nvis=nvis, ncph=min(int(0.3 * nvis), _max_closures(nvis, nsta)), nsta=nsta,
                        nbeta=int(r.integers(16, 49)), nseq=int(r.integers(64, 257))))
    return out


def _points(case, d, seed):
    """Parameter rows over the prior box, or near the truth as a fit's best chains are."""
    r = np.random.default_rng(seed)
    lo, hi = synthdata.EHT_PMIN.astype(np.float64), synthdata.EHT_PMAX.astype(np.float64)
    if not case.get("near", True):
        return (lo + (hi - lo) * r.uniform(size=(case["points"], 9))).astype(np.float32)
    p = d["truth"] + 0.01 * (hi - lo) * r.normal(size=(case["points"], 9))
    return np.clip(p, lo + 1e-3 * (hi - lo), hi - 1e-3 * (hi - lo)).astype(np.float32)


def _fit_of(case, seed):
    b, s, nburn, niter = case["nbeta"], case["nseq"], case["nburn"], case["niter"]
    if case["model"] == "rosenbrock":
        return Fit([1, 1], [-5, -5], [5, 5], np.zeros(1, np.float32), [0.0], [1.0], nbeta=b, nseq=s, nburn=nburn,
                   niter=niter, model="user", npass=1, seed=seed, pstp=0.5, adapt_target=0.25,
                   beta=np.geomspace(1.0, 1e-3, b).astype(np.float32)), "search_Rosenbrock"
    if case["model"] == "solvsys":
        return Fit([1, 1], [-5, -5], [5, 5], np.array([2, 2, 0.25, 0.5], np.float32), [1.0, 0.5], [1.0, 1.0], nbeta=b,
                   nseq=s, nburn=nburn, niter=niter, model="user", npass=1, seed=seed), "solvsys"
    d = _dataset(case["nvis"], case["ncph"], case["nsta"], seed, case["cpext"])
    return _eht_fit(d, case["model"], b, s, seed, nburn, niter), None


def _chi2_inputs(case, seed):
    d = _dataset(case["nvis"], case["ncph"], case["nsta"], seed)
    b, s = case["nbeta"], case["nseq"]
    lo, hi = (synthdata.EHT_PMIN, synthdata.EHT_PMAX) if case["imodel"] == 1 else (P13_MIN, P13_MAX)
    r = np.random.default_rng(seed + 1)
    return d, (lo + (hi - lo) * r.uniform(size=(b, s, lo.size))).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fit":
        fit, project = _fit_of(case, seed)
        lib = os.path.join(ROOT, "examples", project, "libmhre.so") if project else None
        return dict(kind=kind, fit=fit, options=dict(lib=lib, force_generic=case["model"] == "user"))
    if kind == "sample":
        d = _dataset(case["nvis"], case["ncph"], case["nsta"], seed)
        fit = _eht_fit(d, "sgra9", case["nbeta"], case["nseq"], seed, case["nburn"], FOREVER, record=False)
        session = Session([fit], streams=3)
        session.run(case["nburn"])
        return dict(kind=kind, fits=[fit], session=session, iters=case["iters"])
    if kind == "batch":
        fits = []
        for i, f in enumerate(_layout(case)):
            d = _dataset(f["nvis"], f["ncph"], f["nsta"], seed + 1000 * i)
            fits.append(_eht_fit(d, "sgra9", f["nbeta"], f["nseq"], seed + i, FOREVER, 0, record=False))
        return dict(kind=kind, fits=fits, session=Session(fits), iters=case["iters"])
    if kind == "quad":
        n = case["n"]
        ds = synthdata.quadsys_dataset(nsys=case["nsys"], neq=n, n=n, seed=seed)
        nburn, niter = (FOREVER, 0) if case["burn"] else (30, FOREVER)
        fits = [quadsys.quad_fit(ds["Q"][i], ds["b"][i], ds["c"][i], nbeta=case["nbeta"], nseq=case["nseq"],
                                 nburn=nburn, niter=niter, seed=seed + i, record=False) for i in range(case["nsys"])]
        session = Session(fits)
        session.run(30)
        return dict(kind=kind, fits=fits, session=session, iters=case["iters"])
    if kind == "chi2":
        d, rows = _chi2_inputs(case, seed)
        b, s, ndat = case["nbeta"], case["nseq"], case["nvis"] + case["ncph"]
        return dict(kind=kind, imodel=case["imodel"], d=d, pcur=rows, b=b, s=s, ndat=ndat,
                    icoor=d["icoor"] if case["ncph"] else np.zeros(1, np.int32),
                    idat=np.array([case["nvis"], b * s * ndat, 0], np.int32),
                    datm=np.zeros(b * s * (ndat + case["nvis"]), np.float32),
                    chi2m=np.zeros((b, s, ndat), np.float32), chi2c=np.zeros((b, s), np.float32),
                    flag=np.ones((b, s), np.int32))
    d = _dataset(case["nvis"], case["ncph"], case["nsta"], seed)
    rows = torch.as_tensor(_points(case, d, seed + 1), device="cuda")
    return dict(kind=kind, data=adjoint.EhtData.from_dataset(d), rows=rows.requires_grad_(kind == "grad"))


# ------------------------------------------------------------------------------------------------------------ run

def _chains(fits, names):
    return {k: np.concatenate([getattr(f, k).ravel() for f in fits]) for k in names}


def run(state):
    kind = state["kind"]
    if kind == "fit":
        run_fits([state["fit"]], **state["options"])
        return _chains([state["fit"]], ("pout", "tout", "chi2", "pcur", "chi2c", "tcur", "pstp", "n_cnt", "n_acpt",
                                        "n_exch", "n_hist"))
    if kind in ("sample", "batch", "quad"):
        state["session"].run(state["iters"])
        state["session"].download()
        return _chains(state["fits"], ("pcur", "chi2c", "tcur", "pstp", "n_cnt", "n_acpt", "n_exch"))
    if kind == "grad":
        rows = state["rows"]
        rows.grad = None
        chi2 = adjoint.chi2(rows, state["data"])
        chi2.sum().backward()
        return {"chi2": chi2, "grad": rows.grad}
    if kind == "normal":
        chi2, jtr, jtj = state["data"].gn_system(state["rows"])
        return {"chi2": chi2, "jtr": jtr, "jtj": jtj}
    d, rows = state["d"], state["pcur"]
    mcmc_interf.calcmodchi2(d["coor"], d["dat"], d["std2r"], state["icoor"], state["idat"], state["datm"],
                            state["chi2m"], rows, state["chi2c"], state["flag"], state["imodel"], d["coor"].size,
                            state["ndat"], state["icoor"].size, 3, state["datm"].size, rows.shape[2], state["b"],
                            state["s"])
    return {"chi2c": state["chi2c"], "chi2m": state["chi2m"], "datm": state["datm"]}


# ----------------------------------------------------------------------------------------------------------- work

def _chi2_flops(nvis, ncph, cpext=0):
    return F_VIS * (nvis + (3 * ncph if cpext else 0)) + F_CPH * ncph + F_CHAIN


def _state_bytes(chains, nptot, nprm):
    """pcur, chi2c, tcur, n_exch, pstp, n_cnt, n_acpt and the history (nadj = 100) of every chain."""
    return 4.0 * chains * (nptot + 3 + 3 * nprm + 4 * nprm)


def work(case):
    kind = case["kind"]
    if kind == "fit":
        chains, its = case["nbeta"] * case["nseq"], case["nburn"] + case["niter"]
        nprm = {"rosenbrock": 2, "solvsys": 2, "sgra13": 13}.get(case["model"], 9)
        one = 10.0 if nprm == 2 else _chi2_flops(case["nvis"], case["ncph"], case["cpext"])
        data = 16.0 if nprm == 2 else 20.0 * case["nvis"] + 32.0 * case["ncph"]
        return dict(bytes=2 * _state_bytes(chains, nprm, nprm) + 4.0 * chains * (nprm + 1) * case["niter"] + data,
                    flops=one * nprm * chains * its)
    if kind in ("sample", "batch"):
        fits = _layout(case) if kind == "batch" else [case]
        return dict(bytes=sum(2 * _state_bytes(f["nbeta"] * f["nseq"], 9, 9) + 20.0 * f["nvis"] + 32.0 * f["ncph"]
                              for f in fits),
                    flops=sum(_chi2_flops(f["nvis"], f["ncph"]) * 9 * f["nbeta"] * f["nseq"] * case["iters"]
                              for f in fits))
    if kind == "quad":
        n, chains = case["n"], case["nsys"] * case["nbeta"] * case["nseq"]
        # one moved coordinate: n + 3 multiply-adds per equation
        return dict(bytes=2 * _state_bytes(chains, n, n) + 4.0 * case["nsys"] * n * (n * n + n + 2),
                    flops=2.0 * n * (n + 3) * n * chains * case["iters"])
    nvis, ncph = case["nvis"], case["ncph"]
    data = 20.0 * nvis + 32.0 * ncph
    if kind == "grad":   # the reverse pass costs about two forward passes
        return dict(bytes=data + case["points"] * 80.0, flops=3.0 * case["points"] * _chi2_flops(nvis, ncph))
    if kind == "normal":   # nine tangents, then 54 products per datum
        return dict(bytes=data + case["points"] * (36 + 8 + 72 + 648.0),
                    flops=case["points"] * (3.0 * _chi2_flops(nvis, ncph) + (252 + 108.0) * (nvis + ncph)))
    rows = case["nbeta"] * case["nseq"]
    return dict(bytes=data + 4.0 * rows * (3 * nvis + 2 * ncph + 12), flops=rows * _chi2_flops(nvis, ncph))


# ---------------------------------------------------------------------------------------------------------- exact

UAS2NRAD = PI / 180.0 / 3600.0 * 1e3
GCOEF = 2.0 * (PI / (2.0 * math.sqrt(2.0 * math.log(2.0)))) ** 2


def _bessel_ratio(n, y):
    """J_n(x) / x^n, y = x^2 <= 64, from its power series."""
    k = 40
    c = 1.0 / (2.0 ** n * math.factorial(n))
    t = [c]
    for i in range(1, k):
        t.append(-t[-1] / (4.0 * i * (i + n)))
    s = torch.full_like(y, t[-1])
    for a in reversed(t[:-1]):
        s = s * y + a
    return s


def _ring(U, rho2, Rex, rq, fade, shift):
    """Real and imaginary part of the ring's visibility of unit flux, the inner disk shifted by `shift`."""
    Rin = rq * Rex
    h = (2.0 / PI) / ((Rex ** 2 - Rin ** 2 * (1 + shift / Rex)) * fade + (Rex ** 2 - Rin ** 2 * (1 - shift / Rex)))
    h0 = fade * h
    ye = (2 * PI * Rex) ** 2 * rho2
    yi = rq * rq * ye
    ree = PI * (h + h0) * Rex ** 2 * _bessel_ratio(1, ye)
    ime = -2 * PI ** 2 * (h - h0) * Rex ** 3 * U * _bessel_ratio(2, ye)
    rei = PI * (h + h0 - shift * (h - h0) / Rex) * Rin ** 2 * _bessel_ratio(1, yi)
    imi = -2 * PI ** 2 * (h - h0) * rq * Rin ** 3 * U * _bessel_ratio(2, yi)
    ph = 2 * PI * shift * U
    c, s = torch.cos(ph), torch.sin(ph)
    return ree - (rei * c - imi * s), ime - (rei * s + imi * c)


def _vis(u, v, P):
    """Model visibilities (real, imaginary) [rows, nvis] of 9- or 13-parameter rows."""
    p = [P[:, i:i + 1] for i in range(P.shape[1])]
    if P.shape[1] == 9:
        Zsp, Re, rq, ecc, fade, gax, aq, gq, th = p
        Rex = Re * UAS2NRAD
        shift = ecc * Rex * (1 - rq)
        U = u * torch.cos(th) + v * torch.sin(th)
        gu, gv = U, -u * torch.sin(th) + v * torch.cos(th)
        gph = -2 * PI * (rq * Rex - shift) * U
    else:
        Zsp, Re, rq, ecc, fade, gr, gax, aq, gq, al, be, eta, th = p
        Rex = Re * UAS2NRAD
        shift = ecc * Rex * (1 - rq) * torch.cos(eta - th)
        U = u * torch.cos(th) + v * torch.sin(th)
        gu, gv = u * torch.cos(be) + v * torch.sin(be), -u * torch.sin(be) + v * torch.cos(be)
        gph = -2 * PI * gr * Rex * (u * torch.cos(al) + v * torch.sin(al))
    fx, fy = _ring(U, u * u + v * v, Rex, rq, fade, shift)
    ga = gq * torch.exp(-GCOEF * ((gu * aq * gax * Rex) ** 2 + (gv * gax * Rex) ** 2))
    return Zsp * ((1 - gq) * fx + ga * torch.cos(gph)), Zsp * ((1 - gq) * fy + ga * torch.sin(gph))


def _wrap(x):
    return torch.atan2(torch.sin(x), torch.cos(x))


class _Exact:
    """The observation in 64 bits, from the 32-bit arrays that the framework is given."""

    def __init__(self, d):
        t = lambda a: torch.as_tensor(np.asarray(a), device="cuda").double()   # noqa: E731
        self.nvis, self.ncph = d["nvis"], d["ncph"]
        self.u, self.v = t(d["coor"][0:2 * self.nvis:2]), t(d["coor"][1:2 * self.nvis:2])
        self.dat, self.w = t(d["dat"]), t(d["std2r"])
        self.tri = torch.as_tensor(d["cpix"].astype(np.int64), device="cuda").reshape(-1, 3)

    def model(self, P):
        x, y = _vis(self.u, self.v, P)
        amp, ph = torch.sqrt(x * x + y * y), torch.atan2(y, x)
        cph = _wrap(ph[:, self.tri[:, 0]] + ph[:, self.tri[:, 1]] - ph[:, self.tri[:, 2]])
        return amp, ph, cph

    def residuals(self, P):
        amp, _, cph = self.model(P)
        dif = torch.cat([self.dat[:self.nvis] - amp, _wrap(self.dat[self.nvis:] - cph)], dim=1)
        return dif * torch.sqrt(self.w)


def exact(case, seed):
    kind = case["kind"]
    if kind == "chi2":
        d, rows = _chi2_inputs(case, seed)
        e = _Exact(d)
        P = torch.as_tensor(rows.reshape(-1, rows.shape[2]), device="cuda").double()
        amp, ph, cph = e.model(P)
        term = e.residuals(P) ** 2
        return {"chi2c": term.sum(1).reshape(rows.shape[:2]), "chi2m": term.reshape(*rows.shape[:2], -1),
                "datm": torch.cat([torch.cat([amp, cph], dim=1).ravel(), ph.ravel()])}
    if kind not in ("grad", "normal"):
        return None   # the sampler's decisions: a chain has no value in 64 bits
    d = _dataset(case["nvis"], case["ncph"], case["nsta"], seed)
    e = _Exact(d)
    P = torch.as_tensor(_points(case, d, seed + 1), device="cuda").double()
    step = max(1, 2500000 // case["nvis"])
    if kind == "grad":
        chi2, grad = [], []
        for q in P.split(step):
            q = q.detach().requires_grad_(True)
            c = (e.residuals(q) ** 2).sum(1)
            c.sum().backward()
            chi2.append(c.detach())
            grad.append(q.grad)
        return {"chi2": torch.cat(chi2), "grad": torch.cat(grad)}
    chi2, jtr, jtj = [], [], []
    for q in P.split(step):
        cols = []
        for j in range(9):
            tangent = torch.zeros_like(q)
            tangent[:, j] = 1.0
            r, c = torch.func.jvp(e.residuals, (q,), (tangent,))
            cols.append(c)
        J = torch.stack(cols, dim=2)
        chi2.append((r * r).sum(1))
        jtr.append((J * r[:, :, None]).sum(1))
        jtj.append(torch.stack([(J * J[:, :, j:j + 1]).sum(1) for j in range(9)], dim=2))
    return {"chi2": torch.cat(chi2), "jtr": torch.cat(jtr), "jtj": torch.cat(jtj)}
