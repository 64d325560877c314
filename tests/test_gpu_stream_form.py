"""The factorised forward keeps the moments of a window of buckets on chip and
reduces the other sources from a list.  Populations that make the list empty,
short (staged in one round), of several rounds, and long (windows of its own,
also one bucket beyond the staging space), at the edges of the bins-per-lane
variants (64, 128, 256 bins and one more), with clustered and equal bin
offsets, against the FP64 sum of the plan's interpolant (torch, float64) to
1e-6 of the spectrum's norm: every source is a float weight times an FP64
value, so the error is float rounding (6e-8), not a sum of them."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


def _population(kind, n, seed=3):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = torch.rand(4, n, generator=g, device="cuda", dtype=torch.float64)
    if kind == "narrow":      # a few buckets: no list
        gamma = 30.0 + 0.5 * r[0]
    elif kind == "flat":      # every bucket alike: most sources in the list
        gamma = 10.0 ** (3.0 * r[0])
    elif kind == "two":       # two far apart groups, one bucket of the second
        gamma = torch.where(r[0] < 0.6, 2.0 + 0.01 * r[1], 500.0 + 0 * r[1])
    else:                     # a power law
        gamma = (1.0 + (1e3 ** -1.5 - 1.0) * r[0]) ** (-1 / 1.5)
    if kind == "two":
        c, phi = 0.0 * r[2], 0.0 * r[3]
    else:
        c, phi = 2 * r[2] - 1, 2 * np.pi * r[3]
    s = torch.sqrt(1 - c * c)
    u = (torch.stack([s * torch.cos(phi), s * torch.sin(phi), c]) * gamma).float().contiguous()
    b = torch.zeros(3, n, device="cuda")
    b[2] = 1.0
    return u, b


def _reference(plan, table, u, b, w, e):
    x, y = (a.astype(np.float64) for a in table.nodes())
    K = (len(x) - 1) / np.log2(x[-1] / x[0])
    tau = (np.log2(x) - np.log2(x[0])) * K
    sig = np.diff(y) / np.diff(tau)
    c0, sig = torch.from_numpy(y[:-1] - tau[:-1] * sig).cuda(), torch.from_numpy(sig).cuda()
    bins = torch.from_numpy(plan.bins).cuda().double()
    out = torch.zeros(len(plan.bins), dtype=torch.float64, device="cuda")
    for p in range(0, u.shape[1], 1 << 17):
        q = slice(p, p + (1 << 17))
        ud, bd = u[:, q].double(), b[:, q].double()
        g2 = 1 + (ud * ud).sum(0)
        beta = ud / g2.sqrt()
        v = torch.linalg.cross(beta, bd, dim=0)
        be = 0.0
        if e is not None:
            v, be = v + e[:, q].double(), (beta * e[:, q].double()).sum(0)
        chi = ((v * v).sum(0) - be * be).sqrt()
        t = (torch.log2(bins)[None] - torch.log2(g2 * chi)[:, None] - np.log2(x[0])) * K
        s = t.floor().clamp(0, len(sig) - 1).long()
        F = torch.where((t >= 0) & (t < len(sig)), c0[s] + t * sig[s], torch.zeros_like(t))
        out += (chi if w is None else chi * w[q].double()) @ torch.nan_to_num(F)
    return out * bins


@pytest.mark.parametrize("kind,n,nb,fields", [
    ("narrow", 5000, 64, False), ("narrow", 70001, 256, True), ("power", 1, 200, False), ("power", 1023, 65, True),
    ("power", 1025, 128, False), ("power", 300007, 129, True), ("power", 2000003, 256, False), ("flat", 40000, 1, False),
    ("flat", 262145, 256, True), ("flat", 6000001, 256, False), ("two", 9000001, 256, False),
    ("two", 100003, 200, True), ("power", 300007, 257, False)])
def test_stream_form(kind, n, nb, fields):
    table = T.default_table()
    bins = np.logspace(-2, 6, nb).astype(np.float32) if nb > 1 else np.array([2.0], np.float32)
    if nb == 129:
        bins[64:] = bins[:65]  # equal offsets
    plan = T.SyncPlan(table, bins)
    u, b = _population(kind, n)
    g = torch.Generator(device="cuda").manual_seed(7)
    e = 0.1 * torch.randn(3, n, generator=g, device="cuda") if fields else None
    w = 0.5 + torch.rand(n, generator=g, device="cuda") if fields else None
    got = T.sync_spectrum(plan, u, b, w, e, method="binned").double()
    ref = _reference(plan, table, u, b, w, e)
    assert torch.linalg.norm(got - ref) <= 1e-6 * torch.linalg.norm(ref)
