"""Targets and spectrum staged again: a list or table equal to the staged one
is not uploaded again, any other one is. Every hit table of one context that
changes its inputs between propagations equals, bit for bit, that of a fresh
context with the same inputs."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def table(P, dev, targets, spectrum, seed, config=None):
    src = P.PointlikeIsotropicEmitter(np.float32([1.0, 2.0, 3.0]), 0.0, 200_000)
    host, own = None, dev is None
    if own:
        host, dev = P.make_hit_buffers(capacity=1 << 18)
    if config:
        cfg = P._lib.pp_config()
        lib = P._lib.load_library()
        assert lib.pp_get_config(dev.handle, ctypes.byref(cfg)) == 0
        for k, v in config.items():
            setattr(cfg, k, v)
        assert lib.pp_set_config(dev.handle, ctypes.byref(cfg)) == 0
    hits, n = P.run_photon_prop_no_local_cache([src], targets, P.CascadiaMediumProperties(),
                                               spectrum, seed, P.HostHitBuffer(), dev,
                                               with_ids=True)
    if own:
        dev.close()
    return hits


def test_staged_again_equals_fresh_context(P, gpu_lib):
    grid = P.make_detector_grid(4, 4, 20.0, 20, 5.0, radius=0.4)
    moved = [P.spherical_target(t.shape.position + np.float32([0, 0, 1]), 0.4, t.module_id)
             for t in grid]
    wider = [P.spherical_target(t.shape.position, 0.5, t.module_id) for t in grid]
    one_off = grid[:-1] + [P.spherical_target(grid[-1].shape.position, 0.41, 320)]
    planar = grid[:10] + [P.rectangular_target((5.0, 5.0, 8.0), 4.0, 3.0, 11)]
    medium = P.CascadiaMediumProperties()
    spec = P.make_biased_cherenkov_spectrum(P.pmt_acceptance_curve(), (300.0, 700.0), medium)
    tab = {n: P.make_cuda_spectral_dist(spec.spectral_dist, (300.0, 700.0), n)
           for n in (30, 600, 8000)}
    mono = P.Monochromatic(430.0)
    runs = [(grid, mono), (list(grid), mono), (moved, mono), (grid, tab[600]), (grid, tab[600]),
            (grid, tab[8000]), (grid, mono), (one_off, tab[30]), (grid, tab[30]), (planar, tab[30]),
            (grid, tab[600]), (grid[:5], tab[600]), ([], tab[600]), (wider, tab[600]),
            (wider, mono), (wider, tab[600])]
    _, dev = P.make_hit_buffers(capacity=1 << 18)
    n_hits = []
    with dev:
        for k, (targets, spectrum) in enumerate(runs):
            a = table(P, dev, targets, spectrum, 7 + k % 3)
            b = table(P, None, targets, spectrum, 7 + k % 3)
            n_hits.append(len(a["time"]))
            for c in a:
                assert np.array_equal(a[c], b[c]), (k, c)
        # other cells for the same list
        a = table(P, dev, grid, mono, 7, dict(grid_cell=12.0))
        b = table(P, None, grid, mono, 7)
        assert all(np.array_equal(a[c], b[c]) for c in a)
    assert min(n_hits[:4]) > 100 and n_hits[12] == 0
