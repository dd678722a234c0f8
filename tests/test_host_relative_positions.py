"""Hit positions relative to their module, block by block: the bits of the plain
expression, for whole and ragged blocks and any memory order."""
import numpy as np
import pytest


@pytest.mark.parametrize("n", [0, 1, 7, 8, 9, 8191, 8192, 8193, 20000])
@pytest.mark.parametrize("rows", [8, 8192])
def test_relative_positions(P, n, rows):
    from photonprop import pom
    pos = np.random.default_rng(n).normal(size=(n, 3)) * 100.0
    center, radius = (np.float32(10.1), -20.0, 5.5), 0.3
    want = ((pos - np.asarray(center, np.float64)) / radius).astype(np.float32)
    for p in (pos, np.asfortranarray(pos), np.repeat(pos, 2, axis=0)[::2]):
        got = pom._relative(p, center, radius, rows)
        assert got.dtype == np.float32 and got.flags.c_contiguous
        assert np.array_equal(got, want)
