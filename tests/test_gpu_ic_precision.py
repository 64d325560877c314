"""Single (gamma, e_soft) pairs: the inverse-Compton terms are as near their value
in 64 bits as the reference's own float arithmetic is (its terms, from the
oracle).  Roundings of either side are a few times 6e-8 at random, so over
N pairs the two rms differ by chance by about 1 / sqrt(N); 1 % is allowed at
N = 60000.  Pairs close to the kinematic limit (q > 0.9), where KN falls to zero
and magnifies the rounding of q by 1 / (1 - q), are compared by that measure and in
the Thomson regime alone: there x is small, so that its own rounding, which both
share, does not hide the reference's further three of q (4.7e-8 together)."""
import numpy as np
import pytest
import torch

from ragnar_amd import torch_ops as T

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


@pytest.mark.parametrize("g_log", [True, False])
@pytest.mark.parametrize("regime", [(-8.0, -3.5), (-3.0, 3.0)])
def test_terms_as_precise_as_the_reference(orc, g_log, regime):
    rng = np.random.default_rng(5)
    ours, theirs = [], []
    for _ in range(60):
        g, f, fs = (np.array([v], np.float32) for v in (10 ** rng.uniform(1, 6), rng.uniform(0.5, 2), rng.uniform(0.5, 2)))
        es = (10 ** rng.uniform(*regime) / 4 / g.astype(float)).astype(np.float32)
        G = 4 * float(g[0]) * float(es[0])
        E = np.sort(float(g[0]) * G / (1 + G) * 10 ** rng.uniform(-6, 0, 1000)).astype(np.float32)
        S = T.ic_spectrum(_dev(g), _dev(f), g_log, _dev(es), _dev(fs), _dev(E)).cpu().numpy()
        R = orc.ic_spectrum(g, f, int(g_log), es, fs, E)
        L = np.longdouble
        x = E.astype(L) / g.astype(L)
        gq = x / (1 - x)
        q = gq / (4 * g.astype(L) * es.astype(L))
        kn = 2 * q * np.log(q) + (1 - q) * (1 + 2 * q + 0.5 * gq * gq / (1 + gq))
        exact = f.astype(L) * fs.astype(L) / es.astype(L) * E.astype(L) ** 2 * kn / g.astype(L) ** (1 if g_log else 2)
        k = q < 0.9
        ours.append((S[k] / exact[k] - 1).astype(float))
        theirs.append((R[k] / exact[k] - 1).astype(float))
    a, b = (float(np.sqrt(np.mean(np.concatenate(v) ** 2))) for v in (ours, theirs))
    assert 0 < a <= 1.01 * b, (a, b)


def test_terms_near_the_limit(orc):
    rng = np.random.default_rng(6)
    one = np.ones(1, np.float32)
    ours, theirs = [], []
    for _ in range(60):
        g = np.array([10 ** rng.uniform(1, 6)], np.float32)
        es = (10 ** rng.uniform(-8.0, -3.5) / 4 / g.astype(float)).astype(np.float32)
        G = 4 * float(g[0]) * float(es[0])
        E = np.sort(float(g[0]) * G / (1 + G) * (1 - 10 ** rng.uniform(-3, -1, 1000))).astype(np.float32)
        S = T.ic_spectrum(_dev(g), _dev(one), True, _dev(es), _dev(one), _dev(E)).cpu().numpy()
        R = orc.ic_spectrum(g, one, 1, es, one, E)
        L = np.longdouble
        x = E.astype(L) / g.astype(L)
        gq = x / (1 - x)
        q = gq / (4 * g.astype(L) * es.astype(L))
        kn = 2 * q * np.log(q) + (1 - q) * (1 + 2 * q + 0.5 * gq * gq / (1 + gq))
        exact = E.astype(L) ** 2 * kn / es.astype(L) / g.astype(L)
        ours.append(((S / exact - 1) * (1 - q)).astype(float))
        theirs.append(((R / exact - 1) * (1 - q)).astype(float))
    a, b = (float(np.sqrt(np.mean(np.concatenate(v) ** 2))) for v in (ours, theirs))
    assert 0 < a <= b, (a, b)
