"""Hit tables beyond the one-launch ordering leave the device as columns, 32768
rows a slice: sizes around a slice, sub-ranges, columns left out and Float64 times
against the host-sorted copy, which splits the records row by row."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COLUMNS = dict(position=(np.float32, 3), direction=(np.float32, 3), initial_direction=(np.float32, 3),
               wavelength=(np.float32, 1), time=(np.float32, 1), dist_travelled=(np.float32, 1),
               module_id=(np.int64, 1), n_steps=(np.int32, 1), photon_id=(np.uint64, 1),
               source_ix=(np.int32, 1))


def copy(P, dev, first, n, names, f64):
    cols = {c: np.full((n, w) if w > 1 else n, 77, np.float64 if f64 and c == "time" else t)
            for c, (t, w) in COLUMNS.items()}
    p = [P._lib.fptr(cols[c]) if c in names else None for c in COLUMNS]
    rc = P._lib.load_library().pp_copy_hits(dev.handle, first, n, p[0], p[1], p[2], p[3], p[4],
                                            int(f64), p[5], p[6], p[7], p[8], p[9])
    assert rc == 0
    return cols


@pytest.mark.parametrize("n", [4097, 32767, 32768, 32769, 65536, 100_001])
def test_column_slices(P, gpu_lib, n):
    lib = P._lib.load_library()
    targets = [P.spherical_target((0.0, 0.0, 5.0), 2.0, 1)]
    sources = [P.PencilEmitter(np.float32([0.1 * i, 0.0, 0.0]), np.float32([0, 0, 1]), 0.0, 0.0, k)
               for i, k in enumerate((n // 3, 0, n - n // 3))]
    medium = P.SimpleMediumProperties(500.0, 1e5, 1.35, 0.95, 0.22)
    devs = []
    for order in (0, 1, 2):
        cfg = P._lib.pp_config()
        cfg.deterministic_order = order
        _, dev = P.make_hit_buffers(capacity=n + 5, config=cfg)
        P.processing.stage(dev, targets, medium, P.Monochromatic(450.0))
        n_hits, n_sim = ctypes.c_int64(), ctypes.c_int64()
        rc = lib.pp_propagate(dev.handle, P.processing.sources_to_pod(sources), 3,
                              ctypes.c_uint64(3), 2, 1.0, ctypes.byref(n_hits), ctypes.byref(n_sim))
        assert rc == 0 and n_hits.value > 0.99 * n
        devs.append(dev)
    m = n_hits.value
    for f64 in (False, True):
        for first, k, names in ((0, m, list(COLUMNS)), (7, m - 9, ["time", "module_id", "position"]),
                                (m - 5, 5, list(COLUMNS)), (3, m - 3, ["photon_id"]), (0, m, [])):
            want = copy(P, devs[2], first, k, names, f64)
            got = copy(P, devs[1], first, k, names, f64)
            for c in COLUMNS:
                assert got[c].dtype == want[c].dtype and np.array_equal(got[c], want[c]), c
        # the buffer's own order: the same rows
        want, got = (copy(P, d, 0, m, list(COLUMNS), f64) for d in (devs[2], devs[0]))
        order = np.lexsort((got["photon_id"], got["source_ix"]))
        for c in COLUMNS:
            assert np.array_equal(got[c][order], want[c]), c
    for d in devs:
        d.close()
