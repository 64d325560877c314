"""SynchrotronSpectrumFromDist at the edges of its two kernels (a wave per bin
up to 4096 sources, the forward kernel beyond), of their 512-source and
256-source tiles and of the 8 bins of a block: the spectrum to the bar of the
other tests (1e-5 of the oracle's FromDist in EXACT and FP64 modes), zero for
an empty distribution and for bins that are not positive."""
import numpy as np
import pytest
import torch

from _spectra import assert_spectrum
from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,nb,log", [(1, 1, True), (63, 8, True), (511, 9, False), (512, 200, True), (513, 7, True),
                                       (4096, 65, True), (4097, 65, True), (4097, 512, False)])
def test_from_dist(orc, ng, nb, log):
    rng = np.random.default_rng(ng + nb)
    g = (np.logspace(0, 3, ng) if log and ng > 1 else np.linspace(1, 100, ng)).astype(np.float32)
    f = (g.astype(np.float64) ** -2 * rng.uniform(0.5, 1.5, ng)).astype(np.float32)
    bins = (np.logspace(-2, 6, nb) if nb > 1 else np.array([0.1])).astype(np.float32)
    plan = T.SyncPlan(T.default_table(), bins)
    got = T.sync_fromdist(plan, torch.from_numpy(g).cuda(), torch.from_numpy(f).cuda(), log).cpu().numpy()
    _, ex = orc.sync_fromdist(g, f, log, bins, mode=orc.EXACT, want_fp64=True)
    _, f64 = orc.sync_fromdist(g, f, log, bins, mode=orc.FP64, want_fp64=True)
    assert_spectrum(got, ex, f64, what=f"{ng} sources, {nb} bins")


def test_empty_distribution_and_dead_bins():
    bins = np.array([0.1, 0.0, -1.0, 2.0], np.float32)
    plan = T.SyncPlan(T.default_table(), bins)
    one = torch.full((1,), 3.0, device="cuda")
    got = T.sync_fromdist(plan, one, one, True)
    assert got[0] > 0 and got[3] > 0 and not got[1:3].any()
    lib, out = T.lib(), torch.full((4,), 7.0, device="cuda")
    T.check(lib.rgn_sync_fromdist(plan.handle, one.data_ptr(), one.data_ptr(), 0, 1, out.data_ptr(), None))
    torch.cuda.synchronize()
    assert not out.any()
