"""The automatic launch shape leaves the targets of longer lists in memory and
holds shorter lists in LDS (the line depends on the grid's cells, somewhere
between 320 and 1000 targets); a set block size always holds them in LDS. Hits
are the same, bit for bit, as with a set block size and as with the scan of
every target, in batches and launches per source."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(P, sources, targets, n_steps, search=0, mode=0, block=0):
    cfg = P._lib.pp_config()
    cfg.deterministic_order, cfg.search = 1, search
    cfg.batch_mode, cfg.block_size = mode, block
    host, dev = P.make_hit_buffers(capacity=1 << 20, config=cfg)
    with dev:
        hits, n = P.run_photon_prop_no_local_cache(
            sources, targets, P.CascadiaMediumProperties(), P.Monochromatic(450.0), 3, host, dev,
            n_steps=n_steps, with_ids=True)
    return hits, n


@pytest.mark.parametrize("strings,modules", [(1, 9), (4, 20), (6, 16), (8, 12), (10, 10), (10, 30)])
@pytest.mark.parametrize("n_steps", [0, 1, 2, 15])
def test_target_placement_keeps_hits(P, gpu_lib, strings, modules, n_steps):
    medium = P.CascadiaMediumProperties()
    lp = P.workloads.cascade_params(1e4, medium)
    rng = np.random.default_rng(strings * 100 + modules)
    targets = P.make_detector_grid(strings, strings, 12.0, modules, 5.0, radius=0.8)
    sources = [P.ExtendedCherenkovEmitter(rng.uniform(-8, 8, 3).astype(np.float32),
                                          P.workloads.isotropic_unit(rng), 0.0, n, lp)
               for n in (1, 20_000, 70_001)]
    ref, n_ref = run(P, sources, targets, n_steps, search=P._lib.SEARCH_BRUTE)
    assert n_ref == 90_002 and (n_steps == 0 or len(ref["time"]) > 100)
    for kw in (dict(), dict(block=256), dict(block=1024), dict(mode=P._lib.BATCH_PER_SOURCE),
               dict(mode=P._lib.BATCH_PERSISTENT), dict(mode=P._lib.BATCH_GRAPH)):
        got, n = run(P, sources, targets, n_steps, search=P._lib.SEARCH_GRID, **kw)
        assert n == n_ref, kw
        for c in ref:
            assert np.array_equal(got[c], ref[c]), (kw, c)
