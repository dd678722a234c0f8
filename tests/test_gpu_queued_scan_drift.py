"""The queued scan's box around a small far sphere. A direction of |dir|^2 = 1 + e hits
the sphere within sqrt(r^2 + e d^2) of its centre after d metres, which the box
has to allow for. Beams along x, parallel to the box's faces, pass the sphere at
distances inside its radius, beyond the radius and the box's fixed margin but
inside that widened radius, and outside it; sources whose directions are further off
take the plain scan. The rows are those of the scan that tests every target at
every step, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FAR, RADIUS = 1500.0, 0.3
ULP = 2.0 ** -23


def propagate(P, sources, targets, search, n_steps):
    cfg = P._lib.pp_config()
    cfg.search, cfg.deterministic_order = search, 1
    host, dev = P.make_hit_buffers(capacity=1 << 21, config=cfg)
    medium = P.SimpleMediumProperties(5000.0, 600.0, 1.35, 0.95, 0.22)
    with dev:
        return P.run_photon_prop_no_local_cache(sources, targets, medium, P.Monochromatic(450.0), 9,
                                                host, dev, n_steps=n_steps, with_ids=True)


@pytest.mark.parametrize("n_steps", [1, 8])
@pytest.mark.parametrize("ulps", [-1, 0, 1, 8])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_hits_beyond_the_radius(P, gpu_lib, n_steps, ulps, sign):
    length = np.float32(1.0 + ulps * ULP)
    excess = float(length) ** 2 - 1.0
    reach = np.sqrt(max(RADIUS ** 2 + excess * FAR ** 2, 0.0))  # a short direction narrows it
    targets = [P.spherical_target((sign * FAR, 0.0, 0.0), RADIUS, 1)]
    offsets = [0.1, 0.28, 0.5, 0.55, 0.6, 0.7, 0.75, 1.2, 2.0]
    axis = np.float32([sign * length, 0.0, 0.0])
    sources = [P.PencilEmitter(np.float32([0.0, y, 0.0]), axis, 0.0, 0.0, 300_000) for y in offsets]
    out = [propagate(P, sources, targets, s, n_steps)
           for s in (P._lib.SEARCH_BRUTE, P._lib.SEARCH_AUTO)]
    assert out[0][1] == out[1][1] == 300_000 * len(offsets)
    for c in out[0][0]:
        assert np.array_equal(out[0][0][c], out[1][0][c]), c
    # one step in twelve of 600 m is longer than 1500 m
    first = out[0][0]["n_steps"] == 1
    hits = np.bincount(out[0][0]["source_ix"][first], minlength=len(offsets))
    print(f"excess {excess:.2e}, reach {reach:.3f} m, first-step hits {hits}", flush=True)
    # (the start of the reach is 0.4 mm short of the far side's: 0.01 m either way)
    for y, k in zip(offsets, hits):
        assert k > 10_000 if y < reach - 0.01 else k == 0 or y < reach + 0.01, (y, k)
