"""The automatic every-target scan over queued segments (large launches on lists
of up to eight spheres or with planar targets) against the plain scan, which
PP_SEARCH_BRUTE asks for: the same hits, bit for bit. Where it can go wrong:
targets that fill the sky (photons stop after a batch), a target plane through
the source, spheres around it, targets met from hundreds of metres away (where a
direction's drift from unit length widens the reference's sphere test), media
whose longest step makes the targets' box useless, directions that are not of
unit length, one step, hits in every group (16 held back per wave) and a hit
buffer that overflows."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lists(P):
    rng = np.random.default_rng(8)
    u = lambda: P.workloads.isotropic_unit(rng)  # noqa: E731
    sph = lambda n, lo, hi, r: [P.spherical_target(rng.uniform(lo, hi) * u(), r, i + 1)  # noqa: E731
                                for i in range(n)]
    return dict(
        one=sph(1, 10, 10, 0.3), three=sph(3, 2, 30, 0.5), eight=sph(8, 5, 60, 1.0),
        far=sph(2, 400, 600, 0.3) + sph(2, 150, 200, 0.3),
        sky=[P.spherical_target((0.0, 0.0, 3.0), 2.9, 1)],
        around=[P.spherical_target((0.1, 0.0, 0.0), 1.0, 1), P.spherical_target((0.0, 0.0, 0.0), 5.0, 2)],
        plane=[P.rectangular_target((1.0, 0.0, 0.0), 1.0, 4.0, 1)],
        disc=[P.circular_target((0.0, 0.0, 0.0), 2.0, 1), P.circular_target((0.0, 3.0, 8.0), 1.5, 2)],
        mixed=[f(rng.uniform(3, 15) * u(), i) for i in range(1, 9) for f in (
            lambda p, i: P.rectangular_target(p, 3.0, 2.0, 3 * i),
            lambda p, i: P.circular_target(p, 1.2, 3 * i + 1),
            lambda p, i: P.spherical_target(p, 0.5, 3 * i + 2))])


def propagate(P, targets, medium, sources, search, n_steps, mode, capacity=1 << 22):
    cfg = P._lib.pp_config()
    cfg.search, cfg.batch_mode, cfg.deterministic_order = search, mode, 1
    host, dev = P.make_hit_buffers(capacity=capacity, config=cfg)
    with dev:
        return P.run_photon_prop_no_local_cache(sources, targets, medium, P.Monochromatic(450.0), 7,
                                                host, dev, n_steps=n_steps, with_ids=True)


@pytest.mark.parametrize("n_steps", [1, 2, 15])
@pytest.mark.parametrize("name", ["one", "three", "eight", "far", "sky", "around", "plane", "disc",
                                  "mixed"])
def test_equals_plain_scan(P, gpu_lib, name, n_steps):
    targets = lists(P)[name]
    n = 2_000_000
    axis = np.float32([0.6, 0.0, 0.8])
    sources = [P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, n // 2 + 13),
               P.PencilEmitter(np.float32([0.0, 0.1, -4.0]), axis, 0.3, 0.0, n // 2)]
    clear = P.SimpleMediumProperties(500.0, 300.0, 1.35, 0.95, 0.22)
    for medium, mode in ((P.CascadiaMediumProperties(), P._lib.BATCH_PERSISTENT),
                         (clear, P._lib.BATCH_GRAPH), (clear, P._lib.BATCH_PER_SOURCE)):
        want, k = propagate(P, targets, medium, sources, P._lib.SEARCH_BRUTE, n_steps, mode)
        got, n_sim = propagate(P, targets, medium, sources, P._lib.SEARCH_AUTO, n_steps, mode)
        assert n_sim == k == n + 13
        assert len(want["photon_id"]) or n_steps < 15 or name == "far"
        for c in want:
            assert np.array_equal(got[c], want[c]), c


@pytest.mark.parametrize("sca_len,length", [(1e5, 1.0), (1e7, 1.0), (40.0, 1.5)])
def test_useless_box_and_long_directions(P, gpu_lib, sca_len, length):
    targets = lists(P)["mixed"]
    medium = P.SimpleMediumProperties(500.0, sca_len, 1.35, 0.95, 0.22)
    axis = np.float32(length) * np.float32([0.0, 0.6, 0.8])
    sources = [P.PencilEmitter(np.float32([0, 0, 0]), axis, 0.9, 0.0, 300_000)]
    out = [propagate(P, targets, medium, sources, s, 6, P._lib.BATCH_PERSISTENT)
           for s in (P._lib.SEARCH_BRUTE, P._lib.SEARCH_AUTO)]
    assert out[0][1] == out[1][1] == 300_000
    for c in out[0][0]:
        assert np.array_equal(out[0][0][c], out[1][0][c]), c


@pytest.mark.parametrize("capacity", [5_000, 15, 16, 17, 1])
def test_overflow(P, gpu_lib, capacity):
    lib, photons = P._lib.load_library(), 400_000
    full, _ = propagate(P, lists(P)["mixed"], P.CascadiaMediumProperties(),
                        [P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, photons)],
                        P._lib.SEARCH_BRUTE, 4, P._lib.BATCH_PERSISTENT)
    full = len(full["photon_id"])
    assert full > 10_000
    for mode in (P._lib.BATCH_PERSISTENT, P._lib.BATCH_PER_SOURCE):
        cfg = P._lib.pp_config()
        cfg.batch_mode = mode
        _, dev = P.make_hit_buffers(capacity=capacity, config=cfg)
        with dev:
            P.processing.stage(dev, lists(P)["mixed"], P.CascadiaMediumProperties(),
                               P.Monochromatic(450.0))
            pods = P.processing.sources_to_pod(
                [P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, photons)])
            n_hits, n_sim = ctypes.c_int64(), ctypes.c_int64()
            rc = lib.pp_propagate(dev.handle, pods, 1, ctypes.c_uint64(7), 4, 1.0,
                                  ctypes.byref(n_hits), ctypes.byref(n_sim))
            assert rc == P._lib.PP_ERR_HIT_OVERFLOW and n_hits.value == capacity
            assert capacity <= n_sim.value <= photons - (full - capacity)


@pytest.mark.parametrize("n_targets", [1, 12])  # queued scan, grid
def test_photon_ids_beyond_31_bits(P, gpu_lib, n_targets):
    rng = np.random.default_rng(4)
    targets = [P.spherical_target(12.0 * P.workloads.isotropic_unit(rng), 0.3, i + 1)
               for i in range(n_targets)]
    medium = P.SimpleMediumProperties(500.0, 300.0, 1.35, 0.95, 0.22)
    sources = [P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, (1 << 31) + 40_000_000)]
    out = [propagate(P, targets, medium, sources, s, 1, P._lib.BATCH_PERSISTENT, 1 << 24)
           for s in (P._lib.SEARCH_BRUTE, P._lib.SEARCH_AUTO)]
    assert out[0][0]["photon_id"].max() > 1 << 31
    for c in out[0][0]:
        assert np.array_equal(out[0][0][c], out[1][0][c]), c
