"""The factorised forward's list of sources outside the window, against the FP64
sum of the plan's interpolant to 1e-6 of the spectrum's norm (each source is a
float weight times an FP64 value: float rounding, 6e-8).

Sparse lists: one to a few hundred sources in buckets far below or far above
the window, so that the waves which own those buckets are few and the others
have nothing to store before the rounds begin.

Units: fields and B0 scaled together, with particle weights such that chi w is
an ordinary float while its product with B0 is beyond, or below, a float's
range.  The spectrum is that of the unscaled fields times the weight.

Particles that the reference's float steps drop (a momentum whose square
overflows, a chi that overflows or vanishes as a float) add nothing, as in the
pair-by-pair form.

Ordered stores: every particle counts once, whichever tiles a block's waves
start with (one tile to many, whole and cut)."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T
from test_gpu_stream_form import _population, _reference

pytestmark = pytest.mark.gpu


def _isotropic(gamma, seed=11):
    """u of the given moduli, B = z."""
    n = len(gamma)
    g = torch.Generator(device="cuda").manual_seed(seed)
    c = 2 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64) - 1
    phi = 2 * np.pi * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    s = torch.sqrt(1 - c * c)
    u = (torch.stack([s * torch.cos(phi), s * torch.sin(phi), c]) * torch.as_tensor(gamma, device="cuda")).float()
    b = torch.zeros(3, n, device="cuda")
    b[2] = 1.0
    return u.contiguous(), b


@pytest.mark.parametrize("low,high", [(1, 0), (0, 1), (2, 3), (0, 40), (300, 0), (70, 300)])
@pytest.mark.parametrize("nb", [64, 256])
def test_sparse_list(low, high, nb):
    n = 40009
    rng = np.random.default_rng(low * 1000 + high)
    gamma = 30.0 * 1.5 ** rng.random(n)
    at = rng.permutation(n)[: low + high]
    gamma[at[:low]] = 1.5 * 1.6 ** rng.random(low)
    gamma[at[low:]] = 500.0 * 2.0 ** rng.random(high)
    u, b = _isotropic(gamma)
    table = T.default_table()
    plan = T.SyncPlan(table, np.logspace(-2, 6, nb).astype(np.float32))
    ref = _reference(plan, table, u, b, None, None)
    for _ in range(3):
        got = T.sync_spectrum(plan, u, b, method="binned").double()
        assert torch.linalg.norm(got - ref) <= 1e-6 * torch.linalg.norm(ref)


@pytest.mark.parametrize("b0,weight", [(1e12, 1e27), (1e-20, 1e-22), (1e-12, 1e-28), (1e30, 1.0)])
def test_units_of_the_fields(b0, weight):
    b0 = 2.0 ** round(np.log2(b0))  # exact: the scaled fields are the same multiples of B0
    n = 300007
    u, b = _population("power", n)
    table = T.default_table()
    bins = np.logspace(-2, 6, 256).astype(np.float32)
    plan = T.SyncPlan(table, bins, B0=b0)
    got = T.sync_spectrum(plan, u, b * b0, torch.full((n,), weight, device="cuda"), method="binned").double()
    ref = _reference(plan, table, u, b, None, None) * float(np.float32(weight))
    assert torch.linalg.norm(got - ref) <= 1e-6 * torch.linalg.norm(ref)


def test_particles_outside_the_float_range():
    u, b = _population("power", 6000)
    bins = np.logspace(-2, 6, 200).astype(np.float32)
    # momenta around 2^64, the first float whose square is infinite, one component at a time
    edge = np.float32(2.0 ** 64)
    plan = T.SyncPlan(T.default_table(), bins, g_syn=1e19)
    one = torch.zeros(3, 6000, device="cuda")
    m = torch.tensor(np.array([edge, np.nextafter(edge, np.float32(0)), edge / 8, 1.5 * edge], np.float32), device="cuda")
    i = torch.arange(6000, device="cuda")
    one[i % 3, i] = m[i % 4]
    for un in (one, u / u.norm(dim=0) * float(edge)):
        want = T.sync_spectrum(plan, un, b, method="direct").double()
        got = T.sync_spectrum(plan, un, b, method="binned").double()
        assert 0 < torch.linalg.norm(want)
        assert torch.linalg.norm(got - want) <= 1e-6 * torch.linalg.norm(want)
    # chi beyond, and below, a float's range with e_peak inside it
    for field, b0, g_syn in ((1e38, 1e-3, 1e18), (1e-43, 1e5, 1e-17)):
        plan = T.SyncPlan(T.default_table(), bins, B0=b0, g_syn=g_syn)
        for method in ("direct", "binned"):
            assert not torch.any(T.sync_spectrum(plan, u, b * field, method=method)), (field, method)


@pytest.mark.parametrize("n", [1, 1000, 1024 * 256, 1024 * 256 + 1, 1024 * 256 * 2 - 1, 1024 * 256 * 5 + 77, 6000001])
@pytest.mark.parametrize("order", ["ascending", "descending", "cold first"])
def test_ordered_stores(n, order):
    r = torch.rand(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda", dtype=torch.float64)
    gamma = (1.0 + (1e3 ** -1.5 - 1.0) * r) ** (-1 / 1.5)
    key = {"ascending": gamma, "descending": -gamma, "cold first": (gamma > 1.5).double()}[order]
    u, b = _isotropic(gamma[torch.argsort(key)])
    table = T.default_table()
    plan = T.SyncPlan(table, np.logspace(-2, 6, 256).astype(np.float32))
    got = T.sync_spectrum(plan, u, b, method="binned").double()
    ref = _reference(plan, table, u, b, None, None)
    assert torch.linalg.norm(got - ref) <= 1e-6 * torch.linalg.norm(ref)
