"""Hit columns at the edges of their slices: 16384 rows, 32768 of tables beyond
131072 rows, the last slice of one row and whole, against the host-sorted copy; a
table of one slice before and after a longer one on the same context."""
import ctypes

import numpy as np
import pytest

from test_gpu_hit_columns import COLUMNS, copy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16_383, 16_384, 16_385, 131_072, 131_073, 163_840, 163_841])
def test_slice_edges(P, gpu_lib, n):
    targets = [P.spherical_target((0.0, 0.0, 5.0), 4.9, 1)]
    # a source inside the sphere's rim: every photon of the beam hits
    sources = [P.PencilEmitter(np.float32([0.0, 0.0, 0.0]), np.float32([0, 0, 1]), 0.0, 0.0, n)]
    medium = P.SimpleMediumProperties(500.0, 1e7, 1.35, 0.95, 0.22)
    devs = []
    for order in (1, 2):
        cfg = P._lib.pp_config()
        cfg.deterministic_order = order
        _, dev = P.make_hit_buffers(capacity=n + 5, config=cfg)
        P.processing.stage(dev, targets, medium, P.Monochromatic(450.0))
        h, s = ctypes.c_int64(), ctypes.c_int64()
        assert gpu_lib.pp_propagate(dev.handle, P.processing.sources_to_pod(sources), 1,
                                    ctypes.c_uint64(3), 1, 1.0, ctypes.byref(h), ctypes.byref(s)) == 0
        devs.append(dev)
    # steps of 1e7 m: a photon that stops short of the sphere is one in 2e6
    m = h.value
    assert n - 2 <= m <= n
    names = list(COLUMNS)
    for first, k in ((0, 5000), (0, m), (0, min(m, 16_384)), (m - 1, 1), (1, m - 1)):
        for f64 in (False, True):
            want, got = copy(P, devs[1], first, k, names, f64), copy(P, devs[0], first, k, names, f64)
            for c in COLUMNS:
                assert np.array_equal(got[c], want[c]), (first, k, c)
    for d in devs:
        d.close()
