"""The normal equations at the point counts where a point's waves change.

8 waves a point up to 256 points, then 4, 2 and from 1025 points on 1: the
same fp32 terms in another order of float64 sums, 1e-12 of the largest entry.
"""
import numpy as np
import pytest
import torch

from cuda_mcmc_amd import adjoint, synthdata
from tests.helpers import random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nvis,ncph", [(64, 0), (130, 70), (700, 200)])
def test_normal_equations_by_waves_per_point(nvis, ncph):
    data = adjoint.EhtData.from_dataset(synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, seed=nvis))
    lo, hi = synthdata.EHT_PMIN.astype(np.float64), synthdata.EHT_PMAX.astype(np.float64)
    P = torch.as_tensor(random_params(np.random.default_rng(nvis), lo + 0.05 * (hi - lo), hi - 0.05 * (hi - lo), 2049),
                        device="cuda")
    ref = data.gn_system(P)   # one wave per point
    for n in (1, 256, 257, 512, 513, 1024, 1025):
        for a, b in zip(data.gn_system(P[:n].contiguous()), ref):
            b = b[:n]
            scale = b.abs().reshape(n, -1).max(dim=1).values.reshape([n] + [1] * (b.dim() - 1))
            assert a.shape == b.shape and float(((a - b).abs() / scale).max()) < 1e-12
