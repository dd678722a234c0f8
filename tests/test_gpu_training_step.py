"""The two-launch training step against the layer-by-layer kernels: the same
bits in every gradient, parameter and Adam step, since each number is made of
the same products and sums in the same order. Batches around the 32-row tile,
the 64-row bias chunks and the 256-row slices; input and output widths around
the 32-wide tiles; every supported depth, and a depth beyond them (both paths
then run layer by layer). Losses are sums in an order that differs: relative
2^-20 of a sum of up to 4096 terms of one sign."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def batch(rng, n, n_in):
    x = np.clip(rng.normal(0, 1, (n, n_in)), -3, 3).astype(np.float32)
    lab = np.zeros((n, 66), np.float32)
    lab[:, 0] = rng.uniform(10, 1e4, n)
    lab[:, 2:] = rng.poisson(0.3, (n, 64)) * rng.uniform(0.5, 1.0, (n, 64))
    lab[n // 2, 2:] = 0.0                      # a sample without hits
    lab[0, 2:] = rng.uniform(0.5, 40.0, 64)    # and one with every bin filled
    lab[:, 1] = lab[:, 2:].sum(axis=1)
    return x, lab


@pytest.mark.parametrize("n,n_in,n_out,layers", [
    (1, 8, 10, 4), (31, 8, 10, 4), (33, 8, 10, 4), (65, 8, 10, 4), (257, 8, 10, 4),
    (1000, 8, 10, 4), (4096, 8, 10, 4), (300, 1, 10, 1), (300, 32, 32, 2), (300, 17, 31, 3),
    (700, 8, 10, 5), (700, 8, 10, 6), (700, 8, 10, 7), (9000, 8, 10, 4)])
def test_step_equals_layered(P, gpu_lib, n, n_in, n_out, layers):
    from photonprop import surrogate as S
    rng = np.random.default_rng(n + 7 * layers + n_in)
    x, lab = batch(rng, n, n_in)
    out = []
    for fused in (False, True):
        with S.MLP(n_in=n_in, n_out=n_out, n_layers=layers, max_batch=max(n, n_in), seed=3) as m:
            m.set_fused(fused)
            p = m.get_params()
            p += np.random.default_rng(1).normal(0, 0.02, p.size).astype(np.float32)
            m.set_params(p)
            loss, g = m.loss_grad(x, lab)
            m.adam_step(lr=1e-3, weight_decay=0.01)
            curve = m.train(x, lab, 3, batch=n, seed=5, lr=1e-3, weight_decay=0.01)
            y = m.forward(x)                      # the refreshed packed weights
            _, g2 = m.loss_grad(x, lab)
            out.append((g, m.get_params(), y, g2, np.append(curve, loss)))
    for name, a, b in zip(("gradient", "parameters", "outputs", "gradient after"), *out):
        assert np.array_equal(a, b), (name, np.abs(a - b).max())
    np.testing.assert_allclose(out[1][4], out[0][4], rtol=2.0 ** -20 * max(1.0, np.log2(n)))
