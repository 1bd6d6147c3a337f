"""Quadratic systems in calls of one iteration.

A launch writes a parameter's counters, step size and history word only where
the launch proposed it or changed the word; with one iteration a launch most
parameters have neither.  The state after single calls equals that of one call
of many iterations, bit for bit: short, broken and long histories, and systems
with a fixed coordinate.
"""
import numpy as np
import pytest

from cuda_mcmc_amd import quadsys, synthdata
from cuda_mcmc_amd.engine import Session

pytestmark = pytest.mark.gpu

ARRAYS = ("pcur", "chi2c", "pstp", "n_cnt", "n_acpt", "n_hist", "n_exch", "tcur", "flag", "ptent", "ptentn", "pout",
          "tout", "chi2")


@pytest.mark.parametrize("n,nb,ns,nadj", [(8, 16, 9, 100), (8, 5, 13, 33), (4, 32, 2, 1), (2, 3, 21, 31), (8, 64, 1, 64)])
@pytest.mark.parametrize("rows", [True, False])
def test_single_calls_equal_one_call(monkeypatch, n, nb, ns, nadj, rows):
    if not rows:
        monkeypatch.setenv("MHRE_QUAD_FULL", "1")
    ds = synthdata.quadsys_dataset(nsys=1, neq=n, n=n, seed=n + nb)
    one, many = (quadsys.quad_fit(ds["Q"][0], ds["b"][0], ds["c"][0], nbeta=nb, nseq=ns, nburn=40, niter=20, seed=nb,
                                  record=True, nadj=nadj) for _ in range(2))
    for f, calls in ((one, [60]), (many, [1] * 60)):
        with Session([f]) as s:
            assert s.fit_info(0)["quad_rows"] == rows
            for k in calls:
                s.run(k)
            s.download()
    for k in ARRAYS:
        np.testing.assert_array_equal(getattr(one, k), getattr(many, k), err_msg=k)
