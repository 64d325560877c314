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
