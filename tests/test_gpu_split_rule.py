"""Where a ring+Gaussian session splits its chains over waves.

8 waves a chain up to two chains per compute unit, 4 up to four (six with 16
or more chi^2 terms a lane), 8 up to four where LDS holds two work-groups: on
both sides of each limit the form that runs, and the chains of the one-wave
form bit for bit.
"""
import numpy as np
import pytest
import torch

from cuda_mcmc_amd import synthdata
from cuda_mcmc_amd.engine import Session
from tests.helpers import eht_fit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nvis,ncph,model,per_cu,extra,waves", [
    (256, 0, "sgra9", 2, 0, 8), (256, 0, "sgra9", 2, 1, 4), (256, 0, "sgra9", 4, 0, 4), (256, 0, "sgra9", 4, 1, 1),
    (320, 180, "sgra13", 4, 0, 4), (900, 270, "sgra9", 4, 1, 4), (900, 270, "sgra13", 6, 0, 4),
    (900, 270, "sgra9", 6, 1, 1), (1700, 500, "sgra9", 6, 0, 4), (2000, 600, "sgra9", 2, 1, 8),
    (2000, 600, "sgra9", 4, 0, 8), (2000, 600, "sgra9", 4, 1, 1)])
def test_split_by_chains_per_compute_unit(nvis, ncph, model, per_cu, extra, waves):
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    nseq = per_cu * ncu // 8 + extra
    d = synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, seed=nvis)
    one, got = (eht_fit(d, 8, nseq, nburn=2, niter=2, seed=5, model=model) for _ in range(2))
    for f, opt, want in ((one, dict(waves_per_block=4), 1), (got, {}, waves)):
        with Session([f], **opt) as s:
            assert s.fit_info(0)["chain_split"] == want
            s.run(4)
            s.download()
    for k in ("pcur", "chi2c", "pstp", "n_cnt", "n_acpt", "n_exch", "tcur", "pout", "tout", "chi2"):
        np.testing.assert_array_equal(getattr(one, k), getattr(got, k), err_msg=k)
