"""Launches around the photon counts where a batch changes how it deals its chunks (64,
256 and 768 photons per resident wave) against one launch per source: the same hits,
bit for bit, and every photon counted. The counts are those of 24 and of 28 waves
per CU (six and seven per SIMD: the plain scan, and the grid search and the queued
scan), one photon short of the line and on it; 900 photons per 28 waves are beyond
768 for any number of waves up to 32, so that each search takes items from the
counter in one of its runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(P, sources, targets, search, mode):
    cfg = P._lib.pp_config()
    cfg.deterministic_order, cfg.batch_mode, cfg.search = 1, mode, search
    host, dev = P.make_hit_buffers(capacity=1 << 20, config=cfg)
    with dev:
        return P.run_photon_prop_no_local_cache(sources, targets, P.CascadiaMediumProperties(),
                                                P.Monochromatic(450.0), 5, host, dev, n_steps=5,
                                                with_ids=True)


@pytest.mark.parametrize("line,waves", [(64, 24), (64, 28), (256, 24), (256, 28), (768, 24),
                                        (768, 28), (900, 28)])
@pytest.mark.parametrize("kind", ["plain", "queued", "grid"])
def test_both_sides_of_a_line(P, gpu_lib, kind, line, waves):
    _, n_cu = P.autotune.device_arch()
    search = P._lib.SEARCH_BRUTE if kind == "plain" else P._lib.SEARCH_AUTO
    if kind == "grid":
        targets = P.make_detector_grid(3, 3, 12.0, 10, 4.0, radius=0.8)
    else:
        targets = [P.spherical_target((0.0, 0.0, 6.0), 0.5, 1)]
    pos = np.float32([3.0, 2.0, 1.0])
    for photons in (line * waves * n_cu - 1, line * waves * n_cu):
        sources = [P.PointlikeIsotropicEmitter(pos, 0.0, photons // 3),
                   P.PointlikeIsotropicEmitter(-pos, 0.0, photons - photons // 3)]
        want, n = run(P, sources, targets, search, P._lib.BATCH_PER_SOURCE)
        assert n == photons and len(want["time"]) > 20
        for mode in (P._lib.BATCH_PERSISTENT, P._lib.BATCH_GRAPH):
            got, n = run(P, sources, targets, search, mode)
            assert n == photons, (mode, photons)
            for c in want:
                assert np.array_equal(got[c], want[c]), (mode, photons, c)
