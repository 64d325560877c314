"""Where the automatic choice of the forward method changes over: on both sides
of the measured lines, far enough from them that the slower method costs a tenth
or more there (every index of the population, with and without E).  And the
spectrum of one distribution on both sides of its line, which goes by 64-bin
blocks (1950 sources for one block, 450 more for each further one, up to 4096),
to the bar of the other tests."""
import numpy as np
import pytest
import torch

from _spectra import assert_spectrum
from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,fields,direct,binned", [
    (40, False, 240000, 1100000), (87, False, 240000, 800000), (87, True, 400000, 1000000),
    (128, True, 560000, 1000000), (200, False, 400000, 900000), (256, True, 560000, 1130000),
    (320, False, 560000, 1000000), (512, False, 280000, 500000), (512, True, 280000, 560000)])
def test_forward_line(nb, fields, direct, binned):
    plan = T.SyncPlan(T.default_table(), np.logspace(-2, 7, nb).astype(np.float32))
    for n, expect in ((direct, "forward_kernel"), (binned, "binned_")):
        u = torch.full((3, n), 3.0, device="cuda")
        b = torch.ones(3, n, device="cuda")
        b[2] = 0.0
        names = [name for name, _ in T.spectrum_stages(plan, u, b, None, 0.1 * b if fields else None)]
        assert any(name.startswith(expect) for name in names), (n, names)  # a new scratch buffer is cleared first


@pytest.mark.parametrize("ng,nb", [(1950, 64), (1951, 64), (2400, 65), (2401, 128), (3300, 256), (3301, 200), (4097, 400)])
def test_from_dist_line(orc, ng, nb):
    g = np.logspace(0, 3, ng).astype(np.float32)
    f = (g.astype(np.float64) ** -2 * np.random.default_rng(ng).uniform(0.5, 1.5, ng)).astype(np.float32)
    bins = np.logspace(-2, 6, nb).astype(np.float32)
    plan = T.SyncPlan(T.default_table(), bins)
    got = T.sync_fromdist(plan, torch.from_numpy(g).cuda(), torch.from_numpy(f).cuda(), True).cpu().numpy()
    _, ex = orc.sync_fromdist(g, f, True, bins, mode=orc.EXACT, want_fp64=True)
    _, f64 = orc.sync_fromdist(g, f, True, bins, mode=orc.FP64, want_fp64=True)
    assert_spectrum(got, ex, f64, what=f"{ng} sources, {nb} bins")
