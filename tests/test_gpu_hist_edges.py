"""Energy histograms at their bin edges: momenta on and next to every edge (one
component, the others zero, so that |u|^2 is a single rounded product), zero and
subnormal momenta, and momenta past both ends, for bins from ordinary to where
|u|^2 is subnormal.  Counts equal the oracle's; sums agree to 1e-6."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,hi,nb", [
    (-2, 3, 200), (-2, 3, 2741), (0, 0.02, 300), (-20, -18, 50), (-21, -15, 200), (-19.5, 3, 400),
    (-22.2, -18.9, 30), (-18.9, 2, 300), (-30, 30, 500), (-22, -20, 2), (3, 18, 90)])
@pytest.mark.parametrize("fourvel", [True, False])
def test_every_edge(orc, lo, hi, nb, fourvel):
    bins = np.logspace(lo, hi, nb).astype(np.float32)
    plan = T.HistPlan(bins, True)
    e = plan.edges()[1:nb]
    e = e[np.isfinite(e)]
    assert len(e) == nb - 1
    at = np.sqrt(np.maximum(e * e - (0.0 if fourvel else 1.0), 0.0)).astype(np.float32)
    near = [at]
    for _ in range(3):
        near = [np.nextafter(near[0], np.float32(0))] + near + [np.nextafter(near[-1], np.float32(np.inf))]
    past = np.array([0.0, 1e-45, 1e-42, 1e-30, 1e-22, 3e15], np.float32)
    spread = (10.0 ** np.random.default_rng(nb).uniform(max(lo, -23) - 0.5, min(hi, 18) + 0.5, 20 * nb)).astype(np.float32)
    x = np.concatenate(near + [past, spread])
    assert np.isin(at, x).all() and (x == 0).any()
    u = np.zeros((3, len(x)), np.float32)
    u[np.arange(len(x)) % 3, np.arange(len(x))] = x
    h, c = T.energy_hist(plan, torch.from_numpy(u).cuda(), fourvel)
    _, hd, co = orc.energy_hist(u, bins, True, fourvel)
    if fourvel and hi <= 18:
        assert np.count_nonzero(co) > nb // 2
    assert np.array_equal(c.cpu().numpy(), co)
    good = np.isfinite(hd.astype(np.float32))
    h = h.double().cpu().numpy()
    assert np.array_equal(np.isfinite(h), good)
    assert np.all(np.abs(h[good] - hd[good]) <= 1e-6 * np.abs(hd[good]))


@pytest.mark.parametrize("fourvel", [True, False])
def test_terms_are_the_reference_s(fourvel):
    """One particle a bin: each sum is the reference's float term (float)(1 / E), E = sqrtf(|u|^2) or
    sqrt(1 + |u|^2), bit for bit (an FP64 reciprocal of E to about an ulp rounds to the same float except
    within that ulp of a rounding boundary: 1e-9 of the terms)."""
    nb = 2000
    for lo, hi in ((0.2, 3.0), (5.0, 9.0), (-8.0, -6.0) if fourvel else (0.2, 1.0)):
        bins = np.logspace(lo, hi, nb).astype(np.float32)
        plan = T.HistPlan(bins, True)
        for seed in range(10):
            f = np.random.default_rng(seed).uniform(0.2, 0.8, nb - 1)
            e = 10.0 ** (lo + (hi - lo) * (np.arange(nb - 1) + f) / (nb - 1))
            x = np.sqrt(e * e - (0.0 if fourvel else 1.0)).astype(np.float32)
            u = np.zeros((3, nb - 1), np.float32)
            u[seed % 3] = x
            h, c = T.energy_hist(plan, torch.from_numpy(u).cuda(), fourvel)
            assert torch.all(c[:-1] == 1)
            q = x * x
            energy = np.sqrt(q).astype(np.float64) if fourvel else np.sqrt(1.0 + q.astype(np.float64))
            assert np.array_equal(h.cpu().numpy()[:-1], (1.0 / energy).astype(np.float32))
