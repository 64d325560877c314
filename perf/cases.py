"""The framework's workloads as timed cases: sizes, inputs, one pass each.

Every case goes through the public entry points: the torch wrappers of
``ragnar_amd.torch_ops`` (device tensors, plans kept by the caller) or the
drop-in module ``ragnar_amd.ragnar`` (kind "snapshot").  Kinds:

  dist      spectrum of one tabulated distribution (SynchrotronSpectrumFromDist)
  snapshot  a post-processing script's two calls on one particle store through
            the drop-in module: SynchrotronSpectrum_3D and energyDistribution
  spectrum  per-particle spectrum, forward only
  fit       one step of a spectral fit: forward, log-spectrum loss, gradients
            with respect to momenta, fields and weights
  hist      energy histogram of a particle population (counts and sums)
  cells     one spectrum per cell of a ragged particle layout
  rows      many tabulated distributions on one grid, matrix-core contraction
  plaw      the same with the rows given by (index, cutoff)
  ic        inverse-Compton spectrum of two tabulated distributions

``exact`` evaluates the same models in 64 bits with numpy and torch alone.
"""
import math

import numpy as np
import torch

from ragnar_amd import _capi
from ragnar_amd import torch_ops as T

PRECISIONS = {"f16x3": _capi.RGN_PREC_F16X3, "bf16x6": _capi.RGN_PREC_BF16X6}
SIGMA_B = 0.3      # isotropic scatter of the field around B = B0 z
SIGMA_E = 0.1      # electric field, in units of B0
FIT_LOSS = 1.0     # scale of the fit's squared log residuals


def logspace(start, stop, num):
    return np.logspace(math.log10(start), math.log10(stop), num).astype(np.float32)


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def spectrum_case(kind, n, nb, emax=1e7, p=-2.5, e_field=False, weights=False, **more):
    return dict(kind=kind, n=n, nb=nb, emin=1e-2, emax=emax, p=p, e_field=e_field, weights=weights, **more)


def listed():
    return [
        # the smallest call: one distribution on a few hundred bins (latency)
        dict(name="dist-200x200", kind="dist", ng=200, nb=200, gmax=100.0, p=-2.0),
        # a snapshot handled by a reference script, plans made on every call
        dict(name="snapshot-200003", kind="snapshot", n=200003, nb=200, nh=100, p=-2.5),
        # an ordinary population, odd size
        spectrum_case("spectrum", 1000003, 256, name="spectrum-1000003x256"),
        # a population with all fields and weights, as a simulation's output has
        spectrum_case("spectrum", 5000011, 200, e_field=True, weights=True, name="spectrum-fields-5000011x200"),
        # the benchmark's population
        spectrum_case("spectrum", 1 << 24, 256, name="spectrum-16777216x256"),
        # a fit on a small sample (latency of forward, loss and gradients)
        spectrum_case("fit", 30011, 128, emax=1e4, weights=True, name="fit-30011x128"),
        # a fit on a large sample
        spectrum_case("fit", 4000037, 256, emax=1e4, weights=True, name="fit-4000037x256"),
        # the benchmark's histogram
        dict(name="hist-16777216x200", kind="hist", n=1 << 24, nb=200, p=-2.5, fourvel=True, log_bins=True),
        # spatially resolved spectra, ragged cells
        dict(name="cells-4096x256", kind="cells", ncells=4096, median=4000, nb=256),
        # the benchmark's batch of distributions
        dict(name="rows-65536x512x512", kind="rows", nd=65536, ng=512, nb=512, gmax=1e6, precision="f16x3"),
        # a small ragged batch in the mode without a condition on the grid
        dict(name="rows-3001x300x200", kind="rows", nd=3001, ng=300, nb=200, gmax=1e4, precision="bf16x6"),
        # inverse Compton on the reference test's sizes
        dict(name="ic-200x200x200", kind="ic", ng=200, ns=200, ne=200),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["dist", "snapshot", "spectrum", "spectrum", "spectrum", "fit", "fit", "hist", "hist", "cells",
                       "cells", "rows", "rows", "plaw", "ic"])
    p = round(rng.uniform(-3.0, -1.5), 3)
    if kind == "dist":
        return dict(kind=kind, ng=log_int(50, 2000), nb=log_int(20, 500), gmax=10.0 ** rng.randint(2, 5), p=p)
    if kind == "snapshot":
        return dict(kind=kind, n=log_int(1000, 1 << 20), nb=log_int(50, 400), nh=log_int(50, 400), p=p)
    if kind == "spectrum":
        return spectrum_case(kind, log_int(1000, 1 << 24), rng.randint(32, 512), 10.0 ** rng.randint(4, 7), p,
                             rng.random() < 0.4, rng.random() < 0.4)
    if kind == "fit":
        return spectrum_case(kind, log_int(5000, 4000000), rng.randint(32, 384), 10.0 ** rng.randint(2, 3), p,
                             rng.random() < 0.3, rng.random() < 0.8)
    if kind == "hist":
        return dict(kind=kind, n=log_int(10000, 1 << 24), nb=rng.randint(50, 1000), p=p, fourvel=rng.random() < 0.5,
                    log_bins=rng.random() < 0.7)
    if kind == "cells":
        return dict(kind=kind, ncells=log_int(16, 2048), median=log_int(200, 4000), nb=rng.randint(48, 400))
    if kind in ("rows", "plaw"):
        decades = rng.randint(2, 6)
        return dict(kind=kind, nd=log_int(64, 32768), ng=rng.randint(64 * decades, 512), nb=rng.randint(32, 512),
                    gmax=10.0 ** decades, precision=rng.choice(["f16x3", "bf16x6"]))
    return dict(kind=kind, ng=log_int(50, 500), ns=log_int(50, 500), ne=log_int(50, 500))


# ---------------------------------------------------------------------------
# Inputs (made on the GPU from the seed)
# ---------------------------------------------------------------------------
def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def uniform(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def population(g, n, p, e_field=False, weights=False, scale=None, umax=1e3):
    """u, b[, e, w]: |u| a power law of index p on [1, umax] (p may be a tensor
    of n), isotropic; B = z + scatter, times ``scale`` where given."""
    a = 1.0
    b = torch.as_tensor(umax, dtype=torch.float64, device="cuda") ** (p + 1)
    umag = ((b - a) * uniform(g, n) + a) ** (1.0 / (p + 1))
    c = 2.0 * uniform(g, n) - 1.0
    phi = 2.0 * math.pi * uniform(g, n)
    s = torch.sqrt(1.0 - c * c)
    u = torch.stack([s * torch.cos(phi), s * torch.sin(phi), c]).mul_(umag).float()
    B = SIGMA_B * torch.randn(3, n, generator=g, device="cuda")
    B[2] += 1.0
    if scale is not None:
        B *= scale
    e = SIGMA_E * torch.randn(3, n, generator=g, device="cuda") if e_field else None
    w = (0.5 + uniform(g, n)).float() if weights else None
    return u, B, e, w


def cell_layout(case, seed):
    """Lognormal counts; a power-law index and a field scale per cell."""
    rng = np.random.default_rng(seed)
    counts = np.maximum(1, np.round(rng.lognormal(np.log(case["median"]), 1.0, case["ncells"]))).astype(np.int64)
    counts = np.minimum(counts, 40 * case["median"])
    offsets = np.zeros(case["ncells"] + 1, np.int64)
    np.cumsum(counts, out=offsets[1:])
    return offsets, rng.uniform(-3.0, -1.5, case["ncells"]), 10.0 ** rng.uniform(-1.0, 1.0, case["ncells"])


def cell_population(case, seed):
    offsets, p, b0 = cell_layout(case, seed)
    counts = torch.from_numpy(np.diff(offsets)).cuda()
    of = torch.repeat_interleave(torch.arange(case["ncells"], device="cuda"), counts)
    u, b, _, _ = population(generator(seed), int(offsets[-1]), torch.from_numpy(p).cuda()[of],
                            scale=torch.from_numpy(b0).cuda()[of].float())
    return u, b, offsets, of


def dist_inputs(case, seed):
    """A power law with a little scatter on a log grid of gamma beta."""
    g = generator(seed)
    x = torch.from_numpy(logspace(1.0, case["gmax"], case["ng"])).cuda()
    f = x.double() ** case["p"] * torch.exp(0.05 * torch.randn(case["ng"], generator=g, device="cuda").double())
    return x, f.float()


def row_inputs(case, seed):
    """Power laws with exponential cutoffs, each of unit integral."""
    g = generator(seed)
    x = torch.from_numpy(logspace(1.0, case["gmax"], case["ng"])).cuda()
    index = (-3.5 + 2.0 * uniform(g, case["nd"])).float()
    top = math.log10(case["gmax"])
    cutoff = (10.0 ** (top / 3 + top / 2 * uniform(g, case["nd"]))).float()
    return x, index, cutoff


def rows_of(x, index, cutoff):
    xd = x.double()
    f = torch.exp(index.double()[:, None] * torch.log(xd) - xd / cutoff.double()[:, None])
    return f / torch.trapezoid(f, xd)[:, None]


def ic_inputs(case, seed):
    g = generator(seed)
    x = torch.from_numpy(logspace(1e3, 1e7, case["ng"])).cuda()
    s = torch.from_numpy(logspace(1e-11, 1e-7, case["ns"])).cuda()
    k = 0.05 * torch.randn(2, max(case["ng"], case["ns"]), generator=g, device="cuda").double()
    fx = (x.double() ** -2.5 * torch.exp(k[0, : case["ng"]])).float()
    fs = (s.double() ** -1.2 * torch.exp(k[1, : case["ns"]])).float()
    return x, fx, s, fs, torch.from_numpy(logspace(1e-4, 1e7, case["ne"])).cuda()


def photon_bins(case):
    return logspace(case.get("emin", 1e-2), case.get("emax", 1e7), case["nb"])


def fit_target(bins):
    """A smooth target spectrum of the size a fit starts from."""
    x = torch.from_numpy(bins).cuda().double()
    return -0.3 * torch.log(x) - x / 3e4 + 2.0


def hist_bins(case):
    if case["log_bins"]:
        return logspace(1e-2, 1e3, case["nb"])
    return np.linspace(1.0, 100.0, case["nb"]).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "dist":
        s["x"], s["f"] = dist_inputs(case, seed)
        s["plan"] = T.SyncPlan(T.default_table(), photon_bins(case))
    elif kind == "snapshot":
        from ragnar_amd import ragnar as rg

        u, b, e, _ = population(generator(seed), case["n"], case["p"], e_field=True)
        a = {"U": u.cpu().numpy(), "B": b.cpu().numpy(), "E": e.cpu().numpy()}
        prtls = rg.Particles_3D("snapshot")
        prtls.setIgnoreCoords(True)
        prtls.fromArrays({"%s%d" % (q, d + 1): a[q][d] for q in a for d in range(3)})
        s.update(rg=rg, prtls=prtls, bins=rg.Bins(photon_bins(case), rg.EnergyUnits.mec2),
                 hbins=rg.Logbins(1e-1, 1e3, case["nh"]))
    elif kind in ("spectrum", "fit"):
        s["u"], s["b"], s["e"], s["w"] = population(generator(seed), case["n"], case["p"], case["e_field"],
                                                    case["weights"])
        s["plan"] = T.SyncPlan(T.default_table(), photon_bins(case))
        if kind == "fit":
            s["target"] = fit_target(photon_bins(case)).float()
            s["size"] = float(case["n"])
            s["wrt"] = [t.requires_grad_(True) for t in (s["u"], s["b"], s["w"], s["e"]) if t is not None]
    elif kind == "hist":
        s["u"], _, _, _ = population(generator(seed), case["n"], case["p"])
        s["plan"] = T.HistPlan(hist_bins(case), case["log_bins"])
        s["fourvel"] = case["fourvel"]
    elif kind == "cells":
        s["u"], s["b"], s["offsets"], _ = cell_population(case, seed)
        s["plan"] = T.SyncPlan(T.default_table(), photon_bins(case))
    elif kind in ("rows", "plaw"):
        x, index, cutoff = row_inputs(case, seed)
        s["plan"] = T.SyncPlan(T.default_table(), photon_bins(case))
        s.update(x=x, index=index, cutoff=cutoff, precision=PRECISIONS[case["precision"]])
        if kind == "rows":
            s["f"] = rows_of(x, index, cutoff).float()
    elif kind == "ic":
        s["args"] = ic_inputs(case, seed)
    else:
        raise ValueError(kind)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def fit_loss(spectrum, size, target):
    return FIT_LOSS * (torch.log(spectrum / size) - target).square().sum()


def run(s):
    kind = s["kind"]
    if kind == "dist":
        return T.sync_fromdist(s["plan"], s["x"], s["f"], True)
    if kind == "snapshot":
        rg = s["rg"]
        spectrum = rg.SynchrotronSpectrum_3D(s["prtls"], s["bins"], 1.0, 1.0, 1.0)
        return {"spectrum": spectrum.as_array(), "energies": s["prtls"].energyDistribution(s["hbins"]).F().as_array()}
    if kind == "spectrum":
        return T.sync_spectrum(s["plan"], s["u"], s["b"], s["w"], s["e"])
    if kind == "fit":
        spectrum = T.synchrotron_spectrum(s["u"], s["b"], s["w"], s["e"], plan=s["plan"])
        loss = fit_loss(spectrum, s["size"], s["target"])
        return {"spectrum": spectrum.detach(), "grads": torch.autograd.grad(loss, s["wrt"])}
    if kind == "hist":
        return T.energy_hist(s["plan"], s["u"], s["fourvel"])
    if kind == "cells":
        return T.sync_cells(s["plan"], s["u"], s["b"], s["offsets"])
    if kind == "rows":
        return T.sync_fromdist_batched(s["plan"], s["x"], s["f"], True, s["precision"])
    if kind == "plaw":
        return T.sync_fromdist_batched_plaw(s["plan"], s["x"], s["index"], s["cutoff"], True, s["precision"])
    return T.ic_spectrum(*s["args"][:2], True, *s["args"][2:])


def work(case):
    """Inputs read once, outputs written once; operations of the cheapest form
    of the same sum: ~60 per particle for its emission terms, ~60 more for its
    gradients, six per (source, bin) pair of a distribution."""
    kind, nb = case["kind"], case.get("nb", 0)
    n = case.get("n", 0)
    if kind == "dist":
        return {"bytes": 8 * case["ng"] + 4 * nb, "flops": 6 * case["ng"] * nb}
    if kind == "snapshot":
        return {"bytes": (36 + 12) * n + 4 * (nb + case["nh"]), "flops": 80 * n}
    per = 24 + (12 if case.get("e_field") else 0) + (4 if case.get("weights") else 0)
    if kind == "spectrum":
        return {"bytes": per * n + 4 * nb, "flops": 60 * n}
    if kind == "fit":
        return {"bytes": 2 * per * n + 8 * nb, "flops": 120 * n}
    if kind == "hist":
        return {"bytes": 12 * n + 12 * nb, "flops": 12 * n}
    if kind == "cells":
        n = int(case["ncells"] * case["median"] * math.exp(0.5))
        return {"bytes": 24 * n + 4 * case["ncells"] * nb, "flops": 60 * n}
    if kind in ("rows", "plaw"):
        rows = 4 * case["ng"] if kind == "rows" else 8
        return {"bytes": case["nd"] * (rows + 4 * nb), "flops": 2 * case["nd"] * case["ng"] * nb}
    triples = case["ng"] * case["ns"] * case["ne"]
    return {"bytes": 8 * (case["ng"] + case["ns"]) + 8 * case["ne"], "flops": 20 * triples}


# ---------------------------------------------------------------------------
# The same models in 64 bits
# ---------------------------------------------------------------------------
def node_grid(start, stop, num):
    """The reference's float node grid (float exponent, power in double)."""
    f = np.float32
    e = np.log10(f(start)) + np.arange(num, dtype=f) * np.log10(f(stop) / f(start)) / f(num - 1)
    return np.power(10.0, e.astype(np.float64)).astype(f)


def k53(x):
    """K_5/3 by the trapezoid rule on its cosh integral."""
    t = np.arange(0, 1400) / 64.0
    w = np.full(t.size, 1 / 64.0)
    w[0] *= 0.5
    out = np.empty(x.size)
    with np.errstate(over="ignore", under="ignore"):
        for i in range(0, x.size, 1024):
            a = np.minimum(x[i : i + 1024, None] * np.cosh(t), 740.0)
            out[i : i + 1024] = (np.exp(-a) * np.where(a < 740.0, np.cosh(5.0 / 3.0 * np.minimum(t, 400.0)), 0.0)) @ w
    return out


_lines = None


def table_lines():
    """Segments of the reference's 200-node table in t = (log2 x - log2 x_0) K:
    F = c[s] + t sigma[s] on [s, s + 1).  Returns (c, sigma, log2 x_0, K)."""
    global _lines
    if _lines is None:
        x = node_grid(1e-6, 100.0, 200)
        y = np.zeros(200, np.float32)
        for i, xi in enumerate(x):
            if 1e-6 <= xi < 1e-5:
                y[i] = 4 * math.pi / (math.sqrt(3.0) * math.gamma(1 / 3)) * (0.5 * float(xi)) ** (1 / 3)
        mid = [i for i in range(200) if 1e-5 <= x[i] <= 20.0]
        grid = np.stack([node_grid(x[i], 20.0, 100) for i in mid])
        k = k53(grid.astype(np.float64).ravel()).reshape(grid.shape).astype(np.float32)
        total = np.zeros(len(mid), np.float32)
        for m in range(99):  # the reference's float running sum
            step = 0.5 * (k[:, m] + k[:, m + 1]).astype(np.float64) * (grid[:, m + 1] - grid[:, m])
            total = (total.astype(np.float64) + step).astype(np.float32)
        y[mid] = x[mid] * total
        l2 = np.log2(x.astype(np.float64))
        K = 199.0 / np.log2(float(x[-1]) / float(x[0]))
        tau = (l2 - l2[0]) * K
        sigma = np.diff(y.astype(np.float64)) / np.diff(tau)
        c = y[:-1].astype(np.float64) - tau[:-1] * sigma
        _lines = (torch.from_numpy(c).cuda(), torch.from_numpy(sigma).cuda(), float(l2[0]), float(K))
    return _lines


def f_of(t):
    c, sigma, _, _ = table_lines()
    s = t.detach().floor().clamp(0, 198).long()
    return torch.where((t >= 0) & (t < 199), c[s] + t * sigma[s], torch.zeros((), dtype=t.dtype, device=t.device))


def source_terms(u, b, e):
    """chi and the peak energy of every particle (B0 = g_syn = e_at = 1)."""
    gamma2 = 1.0 + (u * u).sum(0)
    beta = u / gamma2.sqrt()
    v = torch.linalg.cross(beta, b, dim=0)
    q = v
    if e is not None:
        q = v + e
        be = (beta * e).sum(0)
        chi = ((q * q).sum(0) - be * be).sqrt()
    else:
        chi = (q * q).sum(0).sqrt()
    return chi, gamma2 * chi


def pair_values(eps, bins):
    _, _, l0, K = table_lines()
    return f_of((torch.log2(bins)[None, :] - torch.log2(eps)[:, None] - l0) * K)


def chunks(n, nb):
    step = max(1, (1 << 26) // nb)
    return [slice(i, min(n, i + step)) for i in range(0, n, step)]


def exact_spectrum(u, b, w, e, bins):
    bins = torch.from_numpy(bins).cuda().double()
    out = torch.zeros(bins.numel(), dtype=torch.float64, device="cuda")
    for c in chunks(u.shape[1], bins.numel()):
        chi, eps = source_terms(u[:, c].double(), b[:, c].double(), None if e is None else e[:, c].double())
        out += (chi if w is None else chi * w[c].double()) @ pair_values(eps, bins)
    return out * bins


def exact_fit(u, b, w, e, bins, size, target):
    spectrum = exact_spectrum(u, b, w, e, bins).requires_grad_(True)
    gout, = torch.autograd.grad(fit_loss(spectrum, size, target.double()), spectrum)
    x = torch.from_numpy(bins).cuda().double()
    grads = [torch.empty(t.shape, dtype=torch.float64, device="cuda") for t in (u, b, w, e) if t is not None]
    for c in chunks(u.shape[1], 4 * x.numel()):
        part = [t[..., c].detach().double().requires_grad_(True) for t in (u, b, w, e) if t is not None]
        named = iter(part)
        uu, bb, ww, ee = (next(named) if t is not None else None for t in (u, b, w, e))
        chi, eps = source_terms(uu, bb, ee)
        loss = (chi if ww is None else chi * ww) @ (pair_values(eps, x) @ (gout * x))
        for g, p in zip(grads, torch.autograd.grad(loss, part)):
            g[..., c] = p
    return {"spectrum": spectrum.detach(), "grads": grads}


def exact_hist(u, bins, fourvel, log_bins):
    usqr = (u.double() ** 2).sum(0)
    energy = usqr.sqrt() if fourvel else (1.0 + usqr).sqrt()
    lo, hi, nb = float(bins.min()), float(bins.max()), len(bins)
    at = ((nb - 1) * (torch.log10(energy / lo).abs() / math.log10(hi / lo))).clamp(0, nb - 1).long()
    at = torch.where(energy < lo, torch.zeros_like(at), torch.where(energy >= hi, torch.full_like(at, nb - 1), at))
    hist = torch.zeros(nb, dtype=torch.float64, device="cuda")
    return hist.index_add_(0, at, 1.0 / energy if log_bins else torch.ones_like(energy))


def exact_cells(u, b, of, ncells, bins):
    bins = torch.from_numpy(bins).cuda().double()
    out = torch.zeros(ncells, bins.numel(), dtype=torch.float64, device="cuda")
    for c in chunks(u.shape[1], bins.numel()):
        chi, eps = source_terms(u[:, c].double(), b[:, c].double(), None)
        out.index_add_(0, of[c], chi[:, None] * pair_values(eps, bins))
    return out * bins


def dist_matrix(x, bins):
    bins = torch.from_numpy(bins).cuda().double()
    return pair_values(x.double() ** 2, bins) * x.double()[:, None] * bins


def exact_ic(x, fx, s, fs, e):
    x, fx, s, fs, e = (t.double() for t in (x, fx, s, fs, e))
    out = torch.empty_like(e)
    G = 4.0 * x[:, None] * s
    top = x[:, None] * G / (1.0 + G)
    for i in range(e.numel()):
        r = e[i] / x[:, None]
        q = r / (G * (1.0 - r))
        qq = torch.where(e[i] <= top, q, torch.ones_like(q))
        kn = 2 * qq * torch.log(qq) + (1 - qq) * (1 + 2 * qq + 0.5 * (G * qq) ** 2 / (1 + G * qq))
        out[i] = (fx[:, None] * (fs / s) * e[i] ** 2 * kn / x[:, None]).sum()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "dist":
        x, f = dist_inputs(case, seed)
        return f.double() @ dist_matrix(x, photon_bins(case))
    if kind == "snapshot":
        u, b, e, _ = population(generator(seed), case["n"], case["p"], e_field=True)
        return {"spectrum": exact_spectrum(u, b, None, e, photon_bins(case)).cpu().numpy(),
                "energies": exact_hist(u, logspace(1e-1, 1e3, case["nh"]), True, True).cpu().numpy()}
    if kind in ("spectrum", "fit"):
        u, b, e, w = population(generator(seed), case["n"], case["p"], case["e_field"], case["weights"])
        if kind == "spectrum":
            return exact_spectrum(u, b, w, e, photon_bins(case))
        return exact_fit(u, b, w, e, photon_bins(case), float(case["n"]), fit_target(photon_bins(case)))
    if kind == "hist":
        u, _, _, _ = population(generator(seed), case["n"], case["p"])
        return exact_hist(u, hist_bins(case), case["fourvel"], case["log_bins"]), None
    if kind == "cells":
        u, b, _, of = cell_population(case, seed)
        return exact_cells(u, b, of, case["ncells"], photon_bins(case))
    if kind in ("rows", "plaw"):
        x, index, cutoff = row_inputs(case, seed)
        f = rows_of(x, index, cutoff)
        return (f.float().double() if kind == "rows" else f) @ dist_matrix(x, photon_bins(case))
    return exact_ic(*ic_inputs(case, seed))
