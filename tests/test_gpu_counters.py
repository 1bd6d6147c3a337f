"""The counts of chi^2 evaluations and proposals (Session.stats).

Every wave adds its counts to the fit once per launch, to one of several
copies where a launch has many waves.  The totals equal the recorded decisions
exactly on every kernel, and the additions do not hold up sessions of many
waves.
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


def _eht(nvis, ncph, nb, ns):
    return eht_fit(synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, seed=5), nb, ns, nburn=3, niter=3, seed=2)


def _rosenbrock(nb, ns, nburn=3, niter=3, **kw):
    return Fit([1, 1], [-5, -5], [5, 5], np.zeros(1, np.float32), [0.0], [1.0], nbeta=nb, nseq=ns, nburn=nburn,
               niter=niter, model="user", npass=1, seed=4, pstp=2.0, record=False, **kw)


def _quad(nb, ns):
    ds = synthdata.quadsys_dataset(nsys=1, neq=4, n=4, seed=6)
    return quadsys.quad_fit(ds["Q"][0], ds["b"][0], ds["c"][0], nbeta=nb, nseq=ns, nburn=3, niter=3, seed=6,
                            record=False)


# one wave a chain (grid and queue), a work-group a chain, whole ladders in a
# wave, lanes of a wave and of a work-group; 1, 2 and more copies, fits side by side
@pytest.mark.parametrize("make,opt", [
    (lambda: [_eht(200, 60, 8, 40)], dict(waves_per_block=4)), (lambda: [_eht(200, 60, 8, 40)], dict(persistent=1)),
    (lambda: [_eht(600, 200, 16, 17), _eht(100, 0, 3, 3)], {}), (lambda: [_quad(16, 700), _quad(5, 7)], {}),
    (lambda: [_quad(70, 150)], {}), (lambda: [_rosenbrock(32, 300)], dict(lib=ROSENBROCK)),
    (lambda: [_rosenbrock(70, 33)], dict(lib=ROSENBROCK)),
    (lambda: [_eht(120, 40, 8, 33)], dict(force_generic=True, graph_iters=2)),
    (lambda: [_eht(300, 90, 8, 17)], dict(force_generic=True, streams=3))])
def test_counts_equal_the_recorded_decisions(make, opt):
    fits = make()
    with Session(fits, trace_iters=6, **opt) as s:
        s.run(4)
        s.run(2)
        s.download()
        st = s.stats()
        traces = [s.trace] if len(fits) == 1 else s.trace
        dec = [t["dec"].copy() for t in traces]
    assert all((d >= 0).all() for d in dec)
    assert st["proposals"] == sum(d.size for d in dec)
    assert st["chi2_evals"] == sum(int(((d >> 8) & 1).sum()) for d in dec)


def test_counting_does_not_hold_up_many_waves():
    """Ladders of 70 rungs, one datum, 8 lanes a chain: 64 sequences are fewer
    waves than the chip holds, 8192 sequences are 9 rounds of its 8192 waves (32
    a compute unit), so they take at most 9 times as long."""
    t = {}
    for ns in (64, 8192):
        with Session([_rosenbrock(70, ns, nburn=4000, niter=0, nadj=8)], lib=ROSENBROCK) as s:
            assert s.fit_info(0)["chain_split"] == 8
            s.run(8)
            t[ns] = 1e30
            for _ in range(5):
                s.run(32)
                s.sync()
                t[ns] = min(t[ns], s.stats()["run_ms"])
    assert t[8192] <= 9 * t[64], t
