"""The inverse-Compton kernel forms a pair's q from per-bin factors and decides
the kinematic limit by q away from it.  Counts at the edges of its stages (128
gamma bins, 512 soft-photon bins, 256 threads), of its chunks and of its row form
(8000 pairs a block, rows three quarters full), and operands
it must leave to the reference's own operations: output energies at and next to
gamma (x = 1), zero output and soft-photon energies, tiny and huge values.

Against the oracle's terms.  KN varies by at most 3 (1 + h) dq / q, h the part
(Gamma q)^2 / (1 + Gamma q) / 2, and either side rounds q to 4 x 6e-8: so each
pair within its limit may differ by 1.5e-6 (1 + h) times its factor (2e-6 is
allowed, and 1e-5 of the sum for the other roundings)."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


def _check(orc, g, fg, g_log, es, fes, E):
    S = T.ic_spectrum(_dev(g), _dev(fg), g_log, _dev(es), _dev(fes), _dev(E)).cpu().numpy()
    _, ex = orc.ic_spectrum(g, fg, int(g_log), es, fes, E, want_fp64=True)
    with np.errstate(all="ignore"):
        assert np.array_equal(np.isnan(S), np.isnan(ex.astype(np.float32)))
        assert np.all(S[ex == 0] == 0)
        G, X = g.astype(float)[None, :, None], E.astype(float)[:, None, None] / g.astype(float)[None, :, None]
        gq = X / (1 - X)
        inside = gq <= 4 * G * es.astype(float) * (1 + 1e-5)
        part = fg[None, :, None] * (fes / es).astype(float) * E[:, None, None].astype(float) ** 2
        part = part / (G if g_log else G * G) * (1 + 0.5 * gq * gq / (1 + gq))
        slack = 2e-6 * np.where(inside & (X < 1), part, 0.0).sum((1, 2))
        ok = np.abs(S - ex) <= 1e-5 * ex + slack
    assert np.all(ok | ~np.isfinite(ex)), (S[~ok][:4], ex[~ok][:4])


@pytest.mark.parametrize("ng,ns,ne", [(1, 1, 60), (128, 1, 40), (129, 3, 40), (127, 255, 30), (257, 256, 7),
                                      (40, 513, 30), (3, 511, 300), (300, 512, 2), (131, 257, 1),
                                      (150, 64, 2100), (130, 560, 1100), (90, 111, 4100)])
@pytest.mark.parametrize("g_log", [True, False])
def test_ic_counts(orc, ng, ns, ne, g_log):
    rng = np.random.default_rng(ng * 1000 + ns)
    g = np.sort(10 ** rng.uniform(0.1, 4, ng)).astype(np.float32)
    es = np.sort(10 ** rng.uniform(-5, 1, ns)).astype(np.float32)
    E = np.sort(10 ** rng.uniform(-4, 4.2, ne)).astype(np.float32)
    _check(orc, g, rng.uniform(0.1, 2, ng).astype(np.float32), g_log, es, rng.uniform(0.1, 2, ns).astype(np.float32), E)


def test_ic_operands(orc):
    g = np.array([1.5, 10.0, 1e3, 1e3 + 1e-3, 2e5, 3e7, 1e13], np.float32)
    es = np.array([0.0, 1e-20, 1e-9, 1e-3, 1.0, 1e4, 1e17], np.float32)
    one = np.ones(7, np.float32)
    E = [0.0, 1e-30, 1e-12, 0.5, 1e14]
    for v in g[1:6]:
        E += [v, np.nextafter(v, np.float32(0)), np.nextafter(v, np.float32(np.inf)), v * (1 - 3e-6), v * (1 - 1e-5),
              v * (1 - 1e-3), v * 1.001]
    E = np.array(sorted(E), np.float32)
    for g_log in (True, False):
        for a, z in ((2, 6), (2, 7), (1, 7)):
            _check(orc, g, one, g_log, es[a:z], one[a:z], E[1:])
        S = T.ic_spectrum(_dev(g), _dev(one), g_log, _dev(es), _dev(one), _dev(E)).cpu().numpy()
        ex = orc.ic_spectrum(g, one, int(g_log), es, one, E)
        assert np.array_equal(np.isnan(S), np.isnan(ex)), (E, S, ex)
