"""Relative positions of short lists need memory of their own size, not of a whole block."""
import tracemalloc

import numpy as np
import pytest


@pytest.mark.parametrize("n", [0, 1, 10, 100, 1000])
def test_short_lists_take_no_whole_block(P, n):
    from photonprop import pom
    pos = np.random.default_rng(n).normal(size=(n, 3))
    center, radius = (10.1, -20.0, 5.5), 0.3
    want = ((pos - np.asarray(center)) / radius).astype(np.float32)
    assert np.array_equal(pom._relative(pos, center, radius), want)
    tracemalloc.start()
    try:
        pom._relative(pos, center, radius)
        peak = tracemalloc.get_traced_memory()[1]
    finally:
        tracemalloc.stop()
    # centres and differences in Float64, the result in Float32: 60 bytes a row, and
    # the objects themselves (a block of 8192 rows takes 200 KB)
    assert peak <= 60 * n + 8192, peak
