"""Launches whose chunks are dealt out by wave index, around the sizes where
the rule changes (64, 256 and 768 photons per resident wave; 6144 waves at six
per SIMD on 256 CUs, fewer with larger tables), against one launch per source:
the same hits, bit for bit, and every photon counted once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(P, sources, targets, spectrum, mode, chunk=0):
    cfg = P._lib.pp_config()
    cfg.deterministic_order, cfg.batch_mode, cfg.chunk_photons = 1, mode, chunk
    host, dev = P.make_hit_buffers(capacity=1 << 20, config=cfg)
    with dev:
        return P.run_photon_prop_no_local_cache(sources, targets, P.CascadiaMediumProperties(),
                                                spectrum, 5, host, dev, n_steps=6, with_ids=True)


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("photons", [1, 63, 65, 1000, 393_215, 393_217, 1_572_863, 1_572_865,
                                     4_718_591, 4_718_593])
def test_dealt_chunks_equal_per_source(P, gpu_lib, photons, split):
    medium = P.CascadiaMediumProperties()
    lp = P.workloads.cascade_params(1e4, medium)
    rng = np.random.default_rng(photons + split)
    counts = [photons - sum(int(photons * f) for f in (0.2, 0.3)[:split - 1])]
    counts += [int(photons * f) for f in (0.2, 0.3)[:split - 1]]
    grid = P.make_detector_grid(3, 3, 30.0, 10, 5.0, radius=1.5)
    one = [P.spherical_target((0.0, 0.0, 6.0), 0.5, 1)]
    for targets, make in (
            (grid, lambda n: P.ExtendedCherenkovEmitter(
                rng.uniform(-20, 20, 3).astype(np.float32), P.workloads.isotropic_unit(rng), 0.0,
                n, lp)),
            (one, lambda n: P.PointlikeIsotropicEmitter(np.zeros(3, np.float32), 0.0, n))):
        sources = [make(n) for n in counts]
        spectrum = P.Monochromatic(450.0)
        ref, n_ref = run(P, sources, targets, spectrum, P._lib.BATCH_PER_SOURCE)
        assert n_ref == photons
        for mode, chunk in ((P._lib.BATCH_PERSISTENT, 0), (P._lib.BATCH_GRAPH, 0),
                            (P._lib.BATCH_PERSISTENT, 64), (P._lib.BATCH_PERSISTENT, 4096)):
            got, n = run(P, sources, targets, spectrum, mode, chunk)
            assert n == photons, (mode, chunk)
            for c in ref:
                assert np.array_equal(got[c], ref[c]), (mode, chunk, c)
