"""What a session reports about its launches.

* time_kernels times the launches that run makes: its step time per iteration,
  also where a launch holds whole sequences for many iterations, is a part of
  run's device time per iteration (1.25 times it for the events between the
  launches), and the iterations advance the chains as run's do.
* autotune times the six launch forms that it can name, and the split form as
  a seventh where a session may take it, each time it is called; the form
  that it returns is one that a session can be given.
* Under a cap on resident waves the exchange launches of one sequence group run
  beside the step launch of another.
"""
import os

import numpy as np
import pytest

from cuda_mcmc_amd import quadsys, synthdata
from cuda_mcmc_amd.engine import Fit, Session
from tests.helpers import eht_fit

pytestmark = pytest.mark.gpu

ROSENBROCK = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "examples",
                          "search_Rosenbrock", "libmhre.so")


def _quad(nfits=1, nburn=600, niter=600):
    ds = synthdata.quadsys_dataset(nsys=nfits, neq=8, n=8, seed=3)
    return [quadsys.quad_fit(ds["Q"][i], ds["b"][i], ds["c"][i], nbeta=16, nseq=32, nburn=nburn, niter=niter, seed=i,
                             record=False) for i in range(nfits)]


def _rosenbrock(nb=32, nburn=600, niter=600):
    return [Fit([1, 1], [-5, -5], [5, 5], np.zeros(1, np.float32), [0.0], [1.0], nbeta=nb, nseq=64, nburn=nburn,
                niter=niter, model="user", npass=1, seed=4, pstp=0.5, record=False)]


def _eht(**kw):
    return [eht_fit(synthdata.ring_gauss_dataset(nvis=323, ncph=100, seed=9), 16, 32, nburn=600, niter=600, seed=1,
                    record=False, **kw)]


@pytest.mark.parametrize("make,lib", [(lambda: _quad(1), None), (lambda: _quad(64), None), (_rosenbrock, ROSENBROCK),
                                      (lambda: _rosenbrock(70), ROSENBROCK), (_eht, None)])
def test_time_kernels_times_the_launches_of_run(make, lib):
    with Session(make(), lib=lib, streams=1) as s:
        s.run(64)
        s.sync()
        step = run = 1e30
        for _ in range(4):
            step = min(step, s.time_kernels(128)[0])
            s.run(128)
            s.sync()
            run = min(run, s.stats()["run_ms"] / 128)
    assert 0 < step <= 1.25 * run, (step, run)


@pytest.mark.parametrize("streams", [1, 3])
def test_time_kernels_advances_the_chains(streams):
    def run(calls):
        fits = _quad(2, nburn=80, niter=60) + _eht()
        fits[2].nburn, fits[2].niter = 70, 90
        with Session(fits, streams=streams) as s:
            for timed, n in calls:
                (s.time_kernels if timed else s.run)(n)
            assert s.stats()["iters_done"] == 140
            s.download()
        return fits
    for a, b in zip(run([(False, 140)]), run([(True, 1), (True, 64), (False, 5), (True, 70)])):
        for k in ("pcur", "chi2c", "pstp", "n_cnt", "n_acpt", "n_hist", "n_exch", "tcur"):
            np.testing.assert_array_equal(getattr(a, k), getattr(b, k), err_msg=k)


@pytest.mark.parametrize("opt,candidates", [({}, 7), (dict(streams=3), 7), (dict(waves_per_block=2), 6),
                                            (dict(persistent=1), 6), (dict(waves_per_simd=2), 6)])
def test_autotune_candidates(opt, candidates):
    ref, got, again = _eht()[0], _eht()[0], _eht()[0]
    with Session([ref]) as s:
        assert s.fit_info(0)["chain_split"] > 1
        s.run(4 * candidates + 5)
        s.download()
    with Session([got], **opt) as s:
        before = s.fit_info(0)["chain_split"]
        assert (before > 1) == (candidates == 7)
        for n in (1, 2):
            w, p, t = s.autotune(2)
            assert w in (1, 2, 4) and p in (0, 1) and t > 0
            assert s.stats()["iters_done"] == 2 * candidates * n
            assert s.fit_info(0)["chain_split"] in (1, before)
        s.run(5)
        s.download()
    with Session([again], waves_per_block=w, persistent=p) as s:   # the named form, not the split one
        assert s.fit_info(0)["chain_split"] == 1
        s.run(4 * candidates + 5)
        s.download()
    for k in ("pcur", "chi2c", "pstp", "n_cnt", "n_acpt", "n_hist", "n_exch", "tcur"):
        np.testing.assert_array_equal(getattr(ref, k), getattr(got, k), err_msg=k)
        np.testing.assert_array_equal(getattr(ref, k), getattr(again, k), err_msg=k)


def test_autotune_where_nothing_can_be_split():
    small = [eht_fit(synthdata.ring_gauss_dataset(nvis=128, ncph=0, seed=9), 4, 4, nburn=60, niter=60, seed=1,
                     record=False)]
    with Session(small) as s:
        s.autotune(2)
        assert s.stats()["iters_done"] == 12


def test_exchange_launches_run_beside_a_capped_step_launch():
    """100 rungs x 40 sequences at 2 waves per SIMD: each of two groups has 2000
    waves of the 2048 that may be resident, so its exchange launch (of ladders
    over 64 rungs, on one lane) costs no time if it runs under the other
    group's step launch; one group has two rounds of waves and its exchange
    after them.  The exchange is about a quarter of the iteration: less than 0.9
    of one group's time if it is hidden, all of it if it waits."""
    d = synthdata.ring_gauss_dataset(nvis=2000, ncph=600, seed=3)
    t = {}
    for streams in (1, 2):
        f = eht_fit(d, 100, 40, nburn=4000, niter=0, seed=1, record=False)
        with Session([f], waves_per_simd=2, streams=streams) as s:
            s.run(32)
            t[streams] = 1e30
            for _ in range(4):
                s.run(32)
                s.sync()
                t[streams] = min(t[streams], s.stats()["run_ms"])
    assert t[2] <= 0.9 * t[1], t
