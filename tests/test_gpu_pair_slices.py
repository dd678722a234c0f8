"""Pair lists at the edges of their slices (65536 pairs with mixtures, 196608 without,
which alternate between two streams) against the same events evaluated in lists of
one slice: the same bits, fused and layer by layer, on one network that lists with
and without mixtures and new weights reach in turn."""
import numpy as np
import pytest

from test_gpu_pair_lists import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [True, False])
def test_slices_equal_single_lists(P, gpu_lib, fused):
    from photonprop import surrogate as S
    dom = S.default_setup().domain()
    rng = np.random.default_rng(6)
    with S.MLP(max_batch=1 << 16, seed=12) as m:
        m.set_fused(fused)
        for n, mixture in ((196_607, False), (65_536, True), (65_537, True), (196_608, False),
                           (196_609, False), (131_072, True), (589_825, False), (200_001, True),
                           (1000, True), (393_216, False)):
            p = m.get_params()
            m.set_params(p + rng.normal(0, 0.02, p.size).astype(np.float32))
            ev, mods = inputs(S, n, 1, n)
            got = m.eval_pairs(ev, mods, dom, mixture=mixture)
            assert got[3] > 0
            for i in range(0, n, 60_000):
                ref = m.eval_pairs(ev[i:i + 60_000], mods, dom, mixture=mixture)
                k = slice(i, i + len(ref[0]))
                assert np.array_equal(got[0][k], ref[0]) and np.array_equal(got[2][k], ref[2]), (n, i)
                assert not mixture or np.array_equal(got[1][k], ref[1]), (n, i)
