"""PMT detection from approximate weights against the full evaluation: the same
PMT for every hit. An acceptance knot below 0 outside the hits' wavelengths
selects the full evaluation and changes nothing else. Widths inside and outside
the range the approximation serves, module orientations (an improper one and
a scaled one, whose cosines leave [-1, 1], among them), hits at the PMT axes and
their antipodes, on the great circles between near and far PMTs, off the
sphere, and non-finite ones."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def ids(P, pom, rel, wl, orient, sigma, seed, full, n_wl=27):
    acc = pom.default_acceptance()
    g = np.linspace(300.0, 820.0, n_wl)
    a1 = np.interp(g, acc.wavelengths, acc.acc_1)
    a2 = np.interp(g, acc.wavelengths, acc.acc_2)
    if full:
        g, a1, a2 = np.append(g, 900.0), np.append(a1, -1.0), np.append(a2, a2[-1])
    else:
        g, a1, a2 = np.append(g, 900.0), np.append(a1, 1.0), np.append(a2, a2[-1])
    model = pom.POMAcceptance(sigma[0], sigma[1], g, a1, a2)
    n = len(rel)
    return pom._pmt_ids(rel, wl, model, orient, np.arange(n) * 977 % (1 << 40),
                        np.arange(n) % 300, seed, 0)


@pytest.mark.parametrize("sigma", [(0.217, 0.290), (0.05, 0.3), (0.021, 0.35), (0.36, 0.37),
                                   (0.4, 0.2), (0.015, 0.3), (1.5, 0.7)])
@pytest.mark.parametrize("orient", ["identity", "rotated", "mirrored", "scaled"])
def test_fast_equals_full(P, gpu_lib, sigma, orient):
    from photonprop import pom
    rot = np.array([[0.36, 0.48, -0.8], [-0.8, 0.6, 0.0], [0.48, 0.64, 0.6]])
    o = dict(identity=None, rotated=rot, mirrored=rot @ np.diag([1.0, 1.0, -1.0]),
             scaled=1.2 * rot)[orient]
    rng = np.random.default_rng(int(1000 * sigma[0]) + len(orient))
    n = 1_500_000
    rel = rng.normal(size=(n, 3))
    rel /= np.linalg.norm(rel, axis=1, keepdims=True)
    d = pom.get_pmt_positions(None, o).astype(np.float64)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    k = n // 8
    near = d[rng.integers(0, 16, k)] + 10.0 ** rng.uniform(-9, -1, (k, 1)) * rng.normal(size=(k, 3))
    rel[:k] = near / np.linalg.norm(near, axis=1, keepdims=True)
    ax = d[rng.integers(0, 16, k)]
    side = np.cross(ax, rng.normal(size=(k, 3)))
    rel[k:2 * k] = side / np.linalg.norm(side, axis=1, keepdims=True)   # c near 0 for one pair
    rel[2 * k:3 * k] *= rng.uniform(0.9, 1.1, (k, 1))
    rel[3 * k:3 * k + 16] = d
    rel[3 * k + 16:3 * k + 20] = [[0, 0, 0], [np.nan, 0, 1], [np.inf, 0, 0], [1e-20, 0, 0]]
    wl = rng.uniform(290, 815, n)
    wl[5:9] = [300.0, 815.0, np.nan, 1e30]
    for seed in (1, 2):
        a = ids(P, pom, rel, wl, o, sigma, seed, False)
        b = ids(P, pom, rel, wl, o, sigma, seed, True)
        bad = np.nonzero(a != b)[0]
        assert len(bad) == 0, (len(bad), bad[:5], rel[bad[:5]], a[bad[:5]], b[bad[:5]])
    assert (b > 0).sum() > 1000


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 524_289])
def test_sizes_and_table_lengths(P, gpu_lib, n):
    from photonprop import pom
    rng = np.random.default_rng(n)
    rel = rng.normal(size=(n, 3))
    rel /= np.linalg.norm(rel, axis=1, keepdims=True)
    wl = rng.uniform(290, 815, n)
    for n_wl in (2, 3, 1023):
        a = ids(P, pom, rel, wl, None, (0.217, 0.29), 5, False, n_wl)
        assert np.array_equal(a, ids(P, pom, rel, wl, None, (0.217, 0.29), 5, True, n_wl))
