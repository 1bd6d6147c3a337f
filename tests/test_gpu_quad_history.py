"""Step-size adaptation of quadratic systems over many iterations per launch.

k_iter_quad carries a parameter's place in its acceptance history and the
counts of its proposals from one proposal to the next and writes n_cnt, n_acpt
and the history back once per launch.  The recorded decisions, replayed here
with the update rule itself (reference: gpu_mcmc.cu:493-522: the rate of the
last min(nadj, n_cnt) outcomes, pstp / 1.01 below the target, else * 1.01),
give the same counters, histories and step sizes exactly: histories shorter
than a launch, of one entry, of whole and broken 32-bit words, and not yet full.
"""
import numpy as np
import pytest

from cuda_mcmc_amd import quadsys, synthdata
from cuda_mcmc_amd.engine import Session

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nadj", [(2, 1), (2, 31), (4, 32), (8, 33), (8, 5), (4, 64), (8, 5000)])
@pytest.mark.parametrize("first", [1, 70])
def test_history_and_counts_replay(n, nadj, first):
    nburn, niter, B, S = 75, 30, 4, 20
    C = B * S
    ds = synthdata.quadsys_dataset(nsys=1, neq=n, n=n, seed=n)
    f = quadsys.quad_fit(ds["Q"][0], ds["b"][0], ds["c"][0], nbeta=B, nseq=S, nburn=nburn, niter=niter, seed=nadj,
                         record=False, nadj=nadj)
    f.n_cnt[:] = first
    pstp = f.pstp.reshape(n, C).copy()
    hist = f.n_hist.reshape(nadj, n, C).copy()
    cnt, acpt = f.n_cnt.reshape(n, C).copy(), f.n_acpt.reshape(n, C).copy()
    with Session([f], trace_iters=nburn + niter) as s:
        s.run(nburn + niter)
        s.download()
        dec = s.trace["dec"].reshape(nburn + niter, n, C).copy()
    sumh, col = hist.sum(axis=0), np.arange(C)
    for it in range(nburn + niter):
        for step in range(n):
            k, acc = dec[it, step] & 0xFF, (dec[it, step] >> 9) & 1
            acpt[k, col] += acc
            if it >= nburn:
                continue
            c, at = cnt[k, col], cnt[k, col] % nadj
            sumh[k, col] += acc - hist[at, k, col]
            hist[at, k, col] = acc
            rate = sumh[k, col].astype(np.float32) / np.minimum(c, nadj).astype(np.float32)
            p = pstp[k, col].astype(np.float64)
            pstp[k, col] = np.where(rate < f.adapt_target, p / 1.01, p * 1.01).astype(np.float32)
            cnt[k, col] = c + 1
    for name, want in (("n_cnt", cnt), ("n_acpt", acpt), ("n_hist", hist), ("pstp", pstp)):
        np.testing.assert_array_equal(getattr(f, name).reshape(want.shape), want, err_msg=name)
