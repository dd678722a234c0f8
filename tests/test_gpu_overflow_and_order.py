"""Counts of a call that overflows its hit buffer, and the order of small hit
tables. An overflowing call completes at least the photons whose hits it stored
and at most those left when every other hit is lost; a call that fits reports
every photon. Tables around the sizes of the one-launch ordering (64 hits per
workgroup, 1024 keys per tile, 4096 hits) equal the host's sort."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def propagate(P, dev, sources, seed=3, n_steps=4):
    lib = P._lib.load_library()
    pods = P.processing.sources_to_pod(sources)
    n_hits, n_sim = ctypes.c_int64(), ctypes.c_int64()
    rc = lib.pp_propagate(dev.handle, pods, len(sources), ctypes.c_uint64(seed), n_steps, 1.0,
                          ctypes.byref(n_hits), ctypes.byref(n_sim))
    return rc, n_hits.value, n_sim.value


@pytest.mark.parametrize("mode", ["PER_SOURCE", "PERSISTENT", "GRAPH"])
@pytest.mark.parametrize("photons", [3_000, 900_000, 12_000_000])
@pytest.mark.parametrize("n_targets", [1, 27])
def test_overflow_counts(P, gpu_lib, mode, photons, n_targets):
    # a target as wide as the source's sky: most photons hit at once
    targets = [P.spherical_target((0.0, 0.0, 3.0), 2.9, 1)]
    targets += [P.spherical_target((40.0 * (i % 5), 30.0, 20.0 * (i // 5)), 0.4, i + 2)
                for i in range(n_targets - 1)]
    cut = photons // 3
    sources = [P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, n)
               for n in (cut, photons - cut)]
    cfg = P._lib.pp_config()
    cfg.batch_mode = getattr(P._lib, "BATCH_" + mode)
    full = None
    for capacity in (1 << 23, 5_000, 7):
        _, dev = P.make_hit_buffers(capacity=capacity, config=cfg)
        with dev:
            P.processing.stage(dev, targets, P.CascadiaMediumProperties(), P.Monochromatic(450.0))
            for _ in range(2):
                rc, n_hits, n_sim = propagate(P, dev, sources)
                if full is None or full <= capacity:
                    full = n_hits
                    assert rc == 0 and n_sim == photons and n_hits > photons // 4
                else:
                    assert rc == P._lib.PP_ERR_HIT_OVERFLOW and n_hits == capacity
                    assert capacity <= n_sim < photons
                    # each photon beyond the stored hits that hits is lost
                    assert n_sim <= photons - (full - capacity)


@pytest.mark.parametrize("n", [0, 1, 2, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 9000])
def test_small_tables_are_ordered(P, gpu_lib, n):
    # every photon hits: three beams into one sphere, which a step of 100 km does not miss
    targets = [P.spherical_target((0.0, 0.0, 5.0), 2.0, 1)]
    parts = [n // 3, 0, n - n // 3]
    sources = [P.PencilEmitter(np.float32([0.1 * i, 0.0, 0.0]), np.float32([0, 0, 1]), 0.0, 0.0, k)
               for i, k in enumerate(parts)]
    out = {}
    for order in (1, 2):
        cfg = P._lib.pp_config()
        cfg.deterministic_order = order
        host, dev = P.make_hit_buffers(capacity=1 << 15, config=cfg)
        with dev:
            out[order], _ = P.run_photon_prop_no_local_cache(
                sources, targets, P.make_simple_medium(30.0, 1e5, 1.35, 0.9, 0.22),
                P.Monochromatic(450.0), 9, host, dev, with_ids=True)
            if order == 1 and len(out[1]["time"]) > 10:  # a later copy of a part
                lib, m = P._lib.load_library(), len(out[1]["time"]) - 7
                pid = np.zeros(m, np.uint64)
                assert lib.pp_copy_hits(dev.handle, 5, m, None, None, None, None, None, 0, None,
                                        None, None, P._lib.fptr(pid), None) == 0
                assert np.array_equal(pid, out[1]["photon_id"][5:5 + m])
    assert n - 3 <= len(out[1]["time"]) <= n
    for c in out[1]:
        assert np.array_equal(out[1][c], out[2][c]), c
