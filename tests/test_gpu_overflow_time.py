"""A call whose hits overflow the buffer ends early, however many photons it asked
for: each wave ends at the first hit that does not fit. A source inside most of its
sky: 1e9 photons into a buffer of 1000 hits against 1e7 photons whose hits fit. A
wave does less than one in a hundred of the large launch, which is what the small
one does; ten times its time is allowed. The photon count stays between the stored
hits and what is left when every other hit is lost."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def propagate(P, targets, photons, capacity, mode, search):
    lib = P._lib.load_library()
    cfg = P._lib.pp_config()
    cfg.batch_mode, cfg.search = mode, search
    _, dev = P.make_hit_buffers(capacity=capacity, config=cfg)
    with dev:
        P.processing.stage(dev, targets, P.CascadiaMediumProperties(), P.Monochromatic(450.0))
        pods = P.processing.sources_to_pod(
            [P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, photons)])
        best = np.inf
        for _ in range(3):
            n_hits, n_sim, ms, k = ctypes.c_int64(), ctypes.c_int64(), ctypes.c_float(), ctypes.c_int32()
            rc = lib.pp_propagate(dev.handle, pods, 1, ctypes.c_uint64(3), 4, 1.0,
                                  ctypes.byref(n_hits), ctypes.byref(n_sim))
            assert lib.pp_last_timing(dev.handle, ctypes.byref(ms), ctypes.byref(k)) == 0
            best = min(best, ms.value)
    return rc, n_hits.value, n_sim.value, best


@pytest.mark.parametrize("mode", ["PER_SOURCE", "PERSISTENT"])
@pytest.mark.parametrize("kind,n_targets", [("BRUTE", 1), ("AUTO", 1), ("GRID", 27)])
def test_overflow_ends_early(P, gpu_lib, mode, kind, n_targets):
    targets = [P.spherical_target((0.0, 0.0, 3.0), 2.9, 1)]
    targets += [P.spherical_target((40.0 * (i % 5), 30.0, 20.0 * (i // 5)), 0.4, i + 2)
                for i in range(n_targets - 1)]
    mode, kind = getattr(P._lib, "BATCH_" + mode), getattr(P._lib, "SEARCH_" + kind)
    rc, hits, n_sim, fits = propagate(P, targets, 10_000_000, 1 << 23, mode, kind)
    assert rc == 0 and n_sim == 10_000_000 and hits > 2_500_000
    share = hits / n_sim
    rc, hits, n_sim, full = propagate(P, targets, 1_000_000_000, 1000, mode, kind)
    print(f"fits {fits:.3f} ms, overflow {full:.3f} ms, {n_sim} photons", flush=True)
    assert rc == P._lib.PP_ERR_HIT_OVERFLOW and hits == 1000
    assert 1000 <= n_sim <= 1_000_000_000 * (1.0 - share) + 1e6
    assert full < 10.0 * fits
