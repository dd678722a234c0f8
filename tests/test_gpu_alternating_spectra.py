"""A driver that alternates between spectra of different lengths (flasher and shower
events on one detector) keeps its grid: a call takes no longer than with one
spectrum by more than half (rebuilding the grid of 3000 targets in every call made it
several times longer). Where the longer spectrum no longer fits beside the grid, the
grid is built again. Hits are those of a fresh context, bit for bit."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spectra(P, knots):
    medium = P.CascadiaMediumProperties()
    spec = P.make_biased_cherenkov_spectrum(P.pmt_acceptance_curve(), (300.0, 700.0), medium)
    return P.make_cuda_spectral_dist(spec.spectral_dist, (300.0, 700.0), knots)


def call(P, dev, pods, n):
    lib = P._lib.load_library()
    h, s = ctypes.c_int64(), ctypes.c_int64()
    assert lib.pp_propagate(dev.handle, pods, n, ctypes.c_uint64(3), 10, 1.0, ctypes.byref(h),
                            ctypes.byref(s)) == 0
    ids, tm = np.zeros(h.value, np.uint64), np.zeros(h.value, np.float32)
    assert lib.pp_copy_hits(dev.handle, 0, h.value, None, None, None, None, P._lib.fptr(tm), 0, None,
                            None, None, P._lib.fptr(ids), None) == 0
    return ids, tm


def context(P):
    cfg = P._lib.pp_config()
    cfg.deterministic_order = 1
    return P.make_hit_buffers(capacity=1 << 18, config=cfg)[1]


@pytest.mark.parametrize("strings,modules", [(10, 30), (6, 10), (16, 30)])
def test_alternating_spectra(P, gpu_lib, strings, modules):
    targets = P.make_detector_grid(strings, strings, 25.0, modules, 6.0, radius=0.5)
    medium = P.CascadiaMediumProperties()
    pods = P.processing.sources_to_pod(
        [P.PointlikeIsotropicEmitter(np.float32([1.0, 2.0, 3.0]), 0.0, 200_000)])
    mono, table = P.Monochromatic(440.0), spectra(P, 600)
    # (the longest spectrum, 32 KB, leaves the grid half of its LDS)
    order = [mono, table, mono, table, spectra(P, 8192), mono]
    with context(P) as dev:
        for s in order:
            P.processing.stage(dev, targets, medium, s)
            got = call(P, dev, pods, 1)
            with context(P) as fresh:
                P.processing.stage(fresh, targets, medium, s)
                want = call(P, fresh, pods, 1)
            assert len(want[0]) > 20
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
    t = {}
    for name, pair in (("one", (table, table)), ("two", (mono, table))):
        times = []
        with context(P) as dev:
            for k in range(40):
                P.processing.stage(dev, targets, medium, pair[k % 2])
                t0 = time.perf_counter()
                call(P, dev, pods, 1)
                times.append(time.perf_counter() - t0)
        t[name] = 1e6 * np.median(times[8:])
    print(f"{len(targets)} targets: one spectrum {t['one']:.0f} us, two {t['two']:.0f} us", flush=True)
    assert t["two"] <= 1.5 * t["one"]
