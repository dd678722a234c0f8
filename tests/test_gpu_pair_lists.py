"""Pair lists around the sizes where the evaluation changes its form: one and
more 32-row tiles, the last list of the small kernel (32 rows per CU, 8192 on
256 CUs), the 128-row tiles, and lists of several slices (2^18 pairs). Hits,
mixtures and flags equal those of the layer-by-layer kernels, whose slices are
other ones (max_batch), bit for bit; pp_mlp_forward likewise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def inputs(S, ne, nm, seed):
    rng = np.random.default_rng(seed)
    ev = np.zeros((ne, 8), np.float32)
    ev[:, :3] = rng.uniform(-300, 300, (ne, 3))
    d = rng.normal(size=(ne, 3))
    ev[:, 3:6] = d / np.linalg.norm(d, axis=1, keepdims=True)
    ev[:, 6] = np.exp(rng.uniform(np.log(20), np.log(5e6), ne))
    ev[:, 7] = rng.uniform(15, 25, ne)
    return ev, rng.uniform(-300, 300, (nm, 3)).astype(np.float32)


@pytest.mark.parametrize("ne,nm,mixture", [
    (1, 1, True), (1, 31, True), (1, 33, True), (8, 1024, True), (2731, 3, True), (16384, 1, True),
    (512, 512, True), (262_145, 1, True), (1, 262_143, False), (700, 1000, True),
    (1000, 787, False)])
def test_lists_equal_layered(P, gpu_lib, ne, nm, mixture):
    from photonprop import surrogate as S
    ev, mods = inputs(S, ne, nm, ne + nm)
    dom = S.default_setup().domain()
    with S.MLP(max_batch=50_000, seed=10) as m:
        p = m.get_params()
        m.set_params(p + np.random.default_rng(2).normal(0, 0.05, p.size).astype(np.float32))
        m.set_fused(False)
        ref = m.eval_pairs(ev, mods, dom, mixture=mixture)
        m.set_fused(True)
        for _ in range(2):  # the second call on the kept workspace
            got = m.eval_pairs(ev, mods, dom, mixture=mixture)
            assert np.array_equal(got[0], ref[0]) and np.array_equal(got[2], ref[2])
            assert not mixture or np.array_equal(got[1], ref[1])
            assert got[3] > 0


@pytest.mark.parametrize("n", [1, 31, 32, 33, 8191, 8192, 8193, 50_000])
@pytest.mark.parametrize("n_in,n_out,layers", [(8, 10, 4), (32, 32, 1), (3, 11, 7)])
def test_forward_equals_layered(P, gpu_lib, n, n_in, n_out, layers):
    from photonprop import surrogate as S
    x = np.random.default_rng(n).normal(0, 1, (n, n_in)).astype(np.float32)
    with S.MLP(n_in=n_in, n_out=n_out, n_layers=layers, max_batch=50_000, seed=4) as m:
        m.set_fused(False)
        ref = m.forward(x)
        m.set_fused(True)
        assert np.array_equal(m.forward(x).view(np.uint32), ref.view(np.uint32))
