"""The model.cuh path at the sizes where a chain's lanes change.

* The number of lanes at exact data counts on both sides of each limit (whole
  ladders in a wave while a lane has at most 4 data, then 8 .. 256 lanes), and
  lock step with the float64 oracle where a fit has at least 60 data.  (The
  lock step's bar, 1e-5 of the chi^2, is one of the sum: a single datum's
  w (d - m)^2 near zero is further off in fp32, 1.6e-3 at a chi^2 of 7e-5.)
* Fits with 2 to 4 data a lane in launches of many iterations: the same chains
  as one iteration a call, from burn-in into sampling, with closures (whose
  second pass reads what other lanes stored in the first).
"""
import numpy as np
import pytest

from cuda_mcmc_amd import synthdata
from cuda_mcmc_amd.engine import Session
from tests.helpers import eht_fit, oracle_eht_chi2
from tests.test_gpu_mhre import _lockstep

pytestmark = pytest.mark.gpu

ARRAYS = ("pcur", "chi2c", "pstp", "n_cnt", "n_acpt", "n_hist", "n_exch", "tcur", "flag", "ptent", "ptentn", "pout",
          "tout", "chi2")


def _data(nvis, ncph, seed=5):
    """The first nvis visibilities of a data set, and ncph closures over any three of them."""
    d = synthdata.ring_gauss_dataset(nvis=max(nvis, 100), ncph=0, seed=seed)
    rng = np.random.default_rng(nvis + ncph)
    tri = np.array([rng.choice(nvis, 3, replace=False) for _ in range(ncph)], np.int32).reshape(-1, 3)
    out = synthdata.pack_eht(d["u"][:nvis], d["v"][:nvis], d["amp"][:nvis], d["eamp"][:nvis],
                             rng.uniform(-3, 3, ncph).astype(np.float32), np.full(ncph, 0.3, np.float32), tri)
    assert out["nvis"] == nvis and out["ncph"] == ncph
    return out


# lanes 64 / 32 rungs = 2 (8 data at most), 64 / 4 = 16 (64), 64 / 1 (256);
# longer ladders or more data: as many lanes as data, 8 to 256
@pytest.mark.parametrize("nvis,ncph,nb,ns,lanes,fused", [
    (1, 0, 32, 3, 2, True), (2, 0, 32, 2, 2, True), (6, 2, 32, 2, 2, True), (7, 2, 32, 2, 16, False),
    (16, 0, 4, 5, 16, True), (60, 4, 4, 9, 16, True), (64, 0, 4, 3, 16, True), (61, 4, 4, 3, 128, False),
    (65, 0, 4, 9, 128, False), (200, 56, 1, 6, 64, True), (201, 56, 1, 6, 256, False), (5, 3, 70, 2, 8, False),
    (30, 2, 70, 2, 32, False), (31, 2, 70, 2, 64, False), (60, 4, 70, 2, 64, False), (124, 4, 70, 2, 128, False),
    (125, 4, 70, 2, 256, False)])
def test_lanes_at_exact_sizes(nvis, ncph, nb, ns, lanes, fused):
    d = _data(nvis, ncph)
    fit = eht_fit(d, nbeta=nb, nseq=ns, nburn=2, niter=2, seed=31 + nb)
    with Session([fit], force_generic=True) as s:
        info = s.fit_info(0)
    assert info["kernel"] == "user" and info["chain_split"] == lanes and info["exchange_in_step"] == fused
    if nvis + ncph >= 60:
        compared, counts = _lockstep(fit, oracle_eht_chi2(d), 4, force_generic=True)
        assert counts["ties"] <= 0.02 * counts["decisions"], counts
        assert compared >= 1


@pytest.mark.parametrize("nvis,ncph,nb,ns,nadj", [
    (3, 0, 32, 5, 100), (6, 2, 32, 3, 33), (24, 8, 8, 7, 100), (60, 4, 4, 5, 3), (200, 56, 1, 3, 100), (13, 2, 16, 9, 31)])
def test_several_data_a_lane_over_many_iterations(nvis, ncph, nb, ns, nadj):
    d = _data(nvis, ncph)

    def run(calls):
        fit = eht_fit(d, nbeta=nb, nseq=ns, nburn=80, niter=70, seed=7, nadj=nadj)
        with Session([fit], force_generic=True) as s:
            info = s.fit_info(0)
            assert info["exchange_in_step"] and info["chain_split"] < nvis + ncph <= 4 * info["chain_split"]
            for n in calls:
                s.run(n)
            s.download()
        return fit
    single = run([1] * 150)
    for calls in ([150], [64, 5, 81]):
        many = run(calls)
        for k in ARRAYS:
            np.testing.assert_array_equal(getattr(single, k), getattr(many, k), err_msg=k)
