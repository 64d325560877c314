"""The pair-by-pair kernels evaluate a source only against the 64-bin blocks it
reaches.  At block, wave and class edges, for sorted and shuffled bins, the
spectrum and the gradients meet the tolerances of the other tests (1e-5 of the
oracle; a summation order is all that changes), and non-finite weights and
upstream gradients still reach every bin and every particle, as when every
pair was evaluated."""
import numpy as np
import pytest
import torch

from _spectra import assert_spectrum, oracle_pair
from ragnar_amd import torch_ops as T
from ragnar_amd import workloads

pytestmark = pytest.mark.gpu


def _case(nb, n, shuffled):
    rng = np.random.default_rng(1000 * nb + n)
    bins = np.logspace(-2, 6, nb).astype(np.float32) if nb > 1 else np.array([0.3], np.float32)
    if shuffled:
        bins = rng.permutation(bins)
    u, b = workloads.particles(n, p=-2.0, seed=nb + n)
    return bins, u, b, rng.uniform(0.5, 2.0, n).astype(np.float32)


@pytest.mark.parametrize("nb,n,shuffled", [(1, 1, False), (64, 63, False), (65, 64, True), (129, 65, False),
                                           (200, 257, True), (256, 5000, False), (320, 700, False),
                                           (448, 300, True), (511, 1000, False), (512, 4097, False)])
def test_blocks_reached(orc, nb, n, shuffled):
    bins, u, b, w = _case(nb, n, shuffled)
    plan = T.SyncPlan(T.default_table(), bins)
    U, B, W = (torch.from_numpy(a).cuda() for a in (u, b, w))
    S = T.sync_spectrum(plan, U, B, W, method="direct")
    ex, f64 = oracle_pair(orc, u, b, bins, w=w)
    assert_spectrum(S.cpu().numpy(), ex, f64, what=f"{nb} bins, {n} particles")
    cells = T.sync_cells(plan, U, B, np.array([0, n // 3, n // 3, n], np.int64), w=W).double().sum(0).cpu().numpy()
    assert np.allclose(cells, S.double().cpu().numpy(), rtol=2e-6, atol=1e-30)

    g = np.random.default_rng(nb).normal(0, 1, nb).astype(np.float32)
    rw, ru, rb, _, dn = orc.sync_adjoint_fp64(u, b, bins, g.astype(np.float64), w=w)
    gw, gu, gb, _ = T.sync_adjoint(plan, U, B, W, None, torch.from_numpy(g).cuda(), need=("w", "u", "b"),
                                   method="direct")
    far = dn >= 1e-4
    for got, ref in ((gw, rw), (gu, ru), (gb, rb)):
        err = np.abs(got.double().cpu().numpy() - ref).reshape(-1, n).max(0)
        assert err[far].max(initial=0.0) <= 1e-5 * max(np.abs(ref).max(), 1e-30)


def test_non_finite_values_reach_every_bin():
    bins, u, b, w = _case(256, 200, False)
    plan = T.SyncPlan(T.default_table(), bins)
    U, B = torch.from_numpy(u).cuda(), torch.from_numpy(b).cuda()
    for bad in (np.nan, np.inf):
        w[70] = bad  # every product with F, zero or not, is then not finite
        S = T.sync_spectrum(plan, U, B, torch.from_numpy(w).cuda(), method="direct")
        assert not torch.isfinite(S).any()
    g = torch.zeros(256, device="cuda")
    g[255] = float("inf")
    gw, _, _, _ = T.sync_adjoint(plan, U, B, None, None, g, need=("w",), method="direct")
    assert not torch.isfinite(gw).any()
