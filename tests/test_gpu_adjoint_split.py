"""Gradient and normal equations with a point's data shared by several waves.

* The gradient's split form (up to 16 waves per point, by the number of points
  and the size of the fit) against the per-closure kernel that
  MHRE_GRAD_RING=0 selects: chi^2 to 1e-6, gradient to 1e-5 of its norm, the
  bars between the other two forms.
* The normal equations of a point do not depend on how many points the call
  holds (1 to 8 waves per point): the same fp32 terms in another order of
  float64 sums, 1e-12 of the largest entry.
"""
import numpy as np
import pytest
import torch

from cuda_mcmc_amd import adjoint, synthdata
from tests.helpers import random_params

pytestmark = pytest.mark.gpu


def _rows(n):
    lo, hi = synthdata.EHT_PMIN.astype(np.float64), synthdata.EHT_PMAX.astype(np.float64)
    span = hi - lo
    return torch.as_tensor(random_params(np.random.default_rng(n), lo + 0.05 * span, hi - 0.05 * span, n), device="cuda")


# tiles: one, one more than one, fewer and more than the waves; no closures;
# closures from points of their own; 16 waves; two rounds; a wave per point
@pytest.mark.parametrize("nvis,ncph,cpext,points", [
    (64, 0, 0, 3), (65, 20, 0, 1), (500, 0, 0, 5), (600, 300, 1, 40), (2100, 600, 0, 300), (2100, 600, 0, 900),
    (1000, 300, 0, 2500), (9000, 2500, 0, 2)])
def test_split_gradient_matches_per_closure_form(monkeypatch, nvis, ncph, cpext, points):
    d = synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, seed=nvis)
    if cpext:
        c = d["cpix"]
        uc = np.stack([d["u"][c[:, 0]], d["v"][c[:, 0]], d["u"][c[:, 1]], d["v"][c[:, 1]]], 1)
        d = dict(d, coor=np.concatenate([d["coor"], uc.ravel()]).astype(np.float32), icoor=None, cpext=1)
    P = _rows(points)
    data = adjoint.EhtData.from_dataset(d)
    chi, g = data.chi2_grad(P)
    only, _ = data.chi2_grad(P, need_grad=False)
    monkeypatch.setenv("MHRE_GRAD_RING", "0")
    chi_c, g_c = data.chi2_grad(P)
    torch.testing.assert_close(chi, chi_c, rtol=1e-6, atol=0)
    torch.testing.assert_close(only, chi_c, rtol=1e-6, atol=0)
    err = (g - g_c).double().norm(dim=1) / g_c.double().norm(dim=1)
    assert float(err.max()) < 1e-5, float(err.max())


@pytest.mark.parametrize("nvis,ncph", [(40, 0), (65, 20), (700, 200)])
def test_normal_equations_do_not_depend_on_the_batch(nvis, ncph):
    d = synthdata.ring_gauss_dataset(nvis=nvis, ncph=ncph, seed=nvis)
    data = adjoint.EhtData.from_dataset(d)
    P = _rows(4100)   # one wave per point
    ref = [x[:7] for x in data.gn_system(P)]
    for n in (7, 513, 1025, 2049):   # 8, 4, 2 and 1 waves per point
        for a, b in zip(data.gn_system(P[:n].contiguous()), ref):
            scale = b.abs().reshape(7, -1).max(dim=1).values.reshape([7] + [1] * (b.dim() - 1))
            assert float(((a[:7] - b).abs() / scale).max()) < 1e-12
