"""The histogram compares |u|^2 with float thresholds instead of forming the
energy.  Counts stay bit-exact against the oracle and sums to 1e-6 (as in the
other histogram tests) for particles on and next to every bin edge, subnormal
and zero momenta, row starts that are not 16-byte aligned (odd n), one and two
bins, bins that start at or below zero energy or repeat one value, and both
energy kinds; NaN and infinite momenta fall in the last bin, as before."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


def _bins(kind, nb):
    return {"log": lambda: np.logspace(-2, 3, nb), "low": lambda: np.logspace(-20, -18, nb),
            "narrow": lambda: np.logspace(0, 0.02, nb), "lin": lambda: np.linspace(1.0, 100.0, nb),
            "zero": lambda: np.linspace(0.0, 50.0, nb), "same": lambda: np.full(nb, 3.0)}[kind]().astype(np.float32)


@pytest.mark.parametrize("kind,nb,log_bins,n", [
    ("log", 200, True, 40001), ("log", 2741, True, 10007), ("log", 1, True, 1), ("log", 2, True, 7),
    ("low", 50, True, 4003), ("narrow", 300, True, 9999), ("lin", 100, False, 30002), ("zero", 64, False, 5001),
    ("same", 5, False, 1025), ("zero", 40, True, 4096)])
@pytest.mark.parametrize("fourvel", [True, False])
def test_thresholds(orc, kind, nb, log_bins, n, fourvel):
    bins = _bins(kind, nb)
    plan = T.HistPlan(bins, log_bins)
    rng = np.random.default_rng(nb + n)
    # momenta along x on both sides of every edge, then a spread past both ends
    e = plan.edges()[1:nb]
    e = e[np.isfinite(e)]
    at = np.sqrt(np.maximum(e * e - (0.0 if fourvel else 1.0), 0.0)).astype(np.float32)
    near = np.concatenate([np.nextafter(at, np.float32(0)), at, np.nextafter(at, np.float32(np.inf))])
    x = np.concatenate([near, np.array([0.0, 1e-42, 1e-30, 3e15], np.float32),
                        (10.0 ** rng.uniform(-3, 4, n)).astype(np.float32)])[-max(n, 1):].astype(np.float32)
    if kind == "same" or kind == "zero":
        x = x[x > 1e-20]
    u = np.zeros((3, len(x)), np.float32)
    u[0] = x
    u[1] = rng.normal(0, 1e-3, len(x)).astype(np.float32) * (rng.random(len(x)) < 0.5)
    h, c = T.energy_hist(plan, torch.from_numpy(u).cuda(), fourvel)
    if kind in ("log", "low", "narrow", "lin"):
        ho, hd, co = orc.energy_hist(u, bins, log_bins, fourvel)
        assert np.array_equal(c.cpu().numpy(), co)
        good = np.isfinite(hd)
        h = h.double().cpu().numpy()
        assert np.array_equal(np.isfinite(h), good)
        assert np.all(np.abs(h[good] - hd[good]) <= 1e-6 * np.maximum(np.abs(hd[good]), 1e-30))
    else:  # one jump, at the largest bin value: everything below is in bin 0
        q = (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]).astype(np.float32)
        en = np.sqrt(q).astype(np.float64) if fourvel else np.sqrt(1.0 + q.astype(np.float64))
        last = int((en >= np.float64(bins.max())).sum())
        want = np.zeros(nb, np.int64)
        want[0], want[-1] = len(x) - last, last
        assert np.array_equal(c.cpu().numpy(), want)


def test_non_finite_momenta():
    plan = T.HistPlan(np.logspace(-2, 3, 200).astype(np.float32), True)
    u = np.ones((3, 9), np.float32)
    u[0, 2], u[1, 5] = np.nan, np.inf
    for counts in (True, False):
        h, c = T.energy_hist(plan, torch.from_numpy(u).cuda(), True, counts=counts)
        assert torch.isnan(h[-1]) and torch.isfinite(h[:-1]).all()
        assert c is None or int(c[-1]) == 2
