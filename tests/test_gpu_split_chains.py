"""One chain over several waves or lanes.

* Ring+Gaussian sessions of few chains run each chain on the waves of a
  work-group (fit_info's chain_split 4 or 8).  The terms of a chi^2 are added
  in the order of the one-wave kernel, so the chains must equal, bit for bit,
  those of a session that names a launch form (waves_per_block = 4: one wave per
  chain).
* The model.cuh path gives a chain 1 to 256 lanes, and runs fits of few data
  in launches of many iterations.  Lock step with the float64 oracle at the
  edges of both, and the same chains whether one call or many run them.
"""
import os

import numpy as np
import pytest

from cuda_mcmc_amd import synthdata
from cuda_mcmc_amd.engine import Fit, Session
from oracle.chi2 import generic_chi2
from tests.helpers import eht_fit, oracle_eht_chi2
from tests.test_gpu_mhre import _lockstep

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ARRAYS = ("pcur", "chi2c", "pstp", "n_cnt", "n_acpt", "n_hist", "n_exch", "tcur", "flag", "ptent", "ptentn", "pout",
          "tout", "chi2")


def _ext(d):
    uv = d["coor"].reshape(-1, 2)
    ext = np.concatenate([uv[d["cpix"][:, 0]], uv[d["cpix"][:, 1]]], axis=1)
    return dict(d, coor=np.concatenate([d["coor"], ext.ravel()]).astype(np.float32))


def _eht(nvis, ncph, model, cpext, nb, ns, nadj=100):
    d = synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, seed=nvis)
    fit = eht_fit(_ext(d) if cpext else d, nb, ns, nburn=9, niter=7, seed=nvis + ncph, model=model, nadj=nadj)
    fit.idat[2] = cpext
    return fit


def _run(fits, segments=(16,), **opt):
    with Session(fits, **opt) as s:
        split = s.fit_info(0)["chain_split"]
        for n in segments:
            s.run(n)
        s.download()
    return split


# one, two and three blocks of 8 tiles (the last shares the blocks among the
# waves), full and partial tiles, no closures, one pass or several per tile,
# closures from points of their own, a history word that fills in a launch
@pytest.mark.parametrize("nvis,ncph,model,cpext,nb,ns,nadj", [
    (256, 0, "sgra9", 0, 8, 4, 100), (257, 1, "sgra9", 0, 5, 3, 33), (323, 319, "sgra9", 0, 32, 16, 100),
    (512, 200, "sgra9", 0, 16, 4, 3), (513, 150, "sgra13", 0, 12, 5, 100), (1100, 900, "sgra9", 0, 8, 8, 100),
    (323, 319, "sgra13", 1, 32, 14, 34), (2000, 600, "sgra9", 0, 32, 8, 100), (640, 64, "sgra9", 0, 70, 2, 100)])
def test_split_chains_bit_identical(nvis, ncph, model, cpext, nb, ns, nadj):
    ref, got = (_eht(nvis, ncph, model, cpext, nb, ns, nadj) for _ in range(2))
    assert _run([ref], waves_per_block=4) == 1
    assert _run([got], segments=(1, 4, 11)) in (4, 8)
    for k in ARRAYS:
        np.testing.assert_array_equal(getattr(ref, k), getattr(got, k), err_msg=k)


def test_split_session_of_uneven_fits_and_its_limits():
    sizes = [(100, 0, 4, 3), (700, 200, 8, 8), (323, 319, 5, 7)]
    ref, got = ([_eht(nv, nc, "sgra9", 0, nb, ns) for nv, nc, nb, ns in sizes] for _ in range(2))
    for f in ref:
        _run([f], waves_per_block=4)
    assert _run(got) in (4, 8)
    for a, b in zip(ref, got):
        for k in ARRAYS:
            np.testing.assert_array_equal(getattr(a, k), getattr(b, k), err_msg=k)
    # too little to share, and more chains than the chip holds work-groups
    assert _run([_eht(128, 0, "sgra9", 0, 4, 4)]) == 1
    assert _run([_eht(323, 100, "sgra9", 0, 32, 256)]) == 1


# the lanes of a chain change at these sizes: whole ladders in a wave (a lane
# per 4 data: 64 / 32 rungs: 2 lanes, 64 / 4: 16), then 8 .. 256 lanes
@pytest.mark.parametrize("nvis,ncph,nb,ns,lanes", [
    (5, 1, 32, 3, 2), (8, 0, 32, 2, 2), (9, 0, 32, 2, 16), (60, 4, 4, 9, 16), (61, 4, 4, 3, 128), (64, 0, 33, 2, 64),
    (120, 8, 3, 2, 128), (200, 56, 3, 2, 256), (300, 90, 70, 2, 256)])
def test_lockstep_model_cuh_lanes(nvis, ncph, nb, ns, lanes):
    d = synthdata.ring_gauss_dataset(nvis=max(nvis, 100), ncph=max(ncph, 0), seed=24)
    if nvis < 100:   # the first records: the closures among them
        keep = (d["cpix"] < nvis).all(axis=1)
        n = min(ncph, int(keep.sum()))
        d = synthdata.pack_eht(d["u"][:nvis], d["v"][:nvis], d["amp"][:nvis], d["eamp"][:nvis], d["cphs"][keep][:n],
                               d["ecph"][keep][:n], d["cpix"][keep][:n])
    fit = eht_fit(d, nbeta=nb, nseq=ns, nburn=2, niter=2, seed=31 + nb)
    with Session([fit], force_generic=True) as s:
        info = s.fit_info(0)
    assert info["kernel"] == "user" and info["chain_split"] == (lanes if d["ncph"] == ncph else info["chain_split"])
    compared, counts = _lockstep(fit, oracle_eht_chi2(d), 4, force_generic=True)
    assert counts["ties"] <= 0.02 * counts["decisions"], counts
    assert compared >= 1


@pytest.mark.parametrize("nb,ns,nadj", [(32, 5, 100), (1, 70, 3), (3, 9, 33), (64, 2, 100), (70, 2, 100)])
def test_model_cuh_iterations_per_launch(nb, ns, nadj):
    def fit():
        return Fit([1, 1], [-5, -5], [5, 5], np.zeros(1, np.float32), [0.0], [1.0], nbeta=nb, nseq=ns, nburn=70,
                   niter=80, model="user", npass=1, seed=nb, pstp=0.5, adapt_target=0.25, nadj=nadj,
                   beta=np.geomspace(1.0, 1e-3, nb).astype(np.float32))
    lib = os.path.join(ROOT, "examples", "search_Rosenbrock", "libmhre.so")
    one, many = fit(), fit()
    _run([one], segments=(150,), lib=lib)
    _run([many], segments=(1, 64, 3, 65, 1, 16), lib=lib)
    for k in ARRAYS:
        np.testing.assert_array_equal(getattr(one, k), getattr(many, k), err_msg=k)
    short = fit()
    short.nburn, short.niter = 2, 2
    short.pout, short.tout, short.chi2 = (np.zeros(x.shape[:-1] + (2,), x.dtype) for x in (one.pout, one.tout, one.chi2))
    f = lambda P: generic_chi2("rosenbrock", P, short.coor, short.dat, short.std2r)   # noqa: E731
    compared, _ = _lockstep(short, f, 4, lib=lib)
    assert compared >= 1


@pytest.mark.parametrize("n,nb,ns,nadj", [(8, 16, 9, 33), (4, 40, 3, 100), (2, 3, 50, 2)])
def test_quadratic_system_iterations_per_launch(n, nb, ns, nadj):
    from cuda_mcmc_amd import quadsys
    ds = synthdata.quadsys_dataset(nsys=1, neq=n, n=n, seed=n)
    one, many = (quadsys.quad_fit(ds["Q"][0], ds["b"][0], ds["c"][0], nbeta=nb, nseq=ns, nburn=70, niter=80, seed=nb,
                                  record=True, nadj=nadj) for _ in range(2))
    _run([one], segments=(150,))
    _run([many], segments=(1, 64, 3, 65, 1, 16))
    for k in ARRAYS:
        np.testing.assert_array_equal(getattr(one, k), getattr(many, k), err_msg=k)
