"""The first evaluation of a pair list by a network costs little more than a later
one, and a list of more than one slice no more than its share. With copies from
device buffers between the slices, the first evaluation of 5e6 pairs took 1.7 times
the later ones, and 3e5 pairs 4.8 times what 1e5 take in one slice, in every call.
The fastest of several fresh networks counts for each call, after one network that
warms the process up."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def evaluate(P, n_events, networks, calls):
    from photonprop import surrogate as S
    rng = np.random.default_rng(n_events)
    ev = np.zeros((n_events, 8), np.float32)
    ev[:, :3] = rng.uniform(-300, 300, (n_events, 3))
    d = rng.normal(size=(n_events, 3))
    ev[:, 3:6] = d / np.linalg.norm(d, axis=1, keepdims=True)
    ev[:, 6], ev[:, 7] = 1e4, 20.0
    mods = rng.uniform(-300, 300, (1000, 3)).astype(np.float32)
    dom = S.default_setup().domain()
    t = np.zeros((networks, calls))
    for i in range(networks):
        with S.MLP(seed=3) as m:
            for k in range(calls):
                t0 = time.perf_counter()
                out = m.eval_pairs(ev, mods, dom)
                t[i, k] = time.perf_counter() - t0
                assert out[3] > 0
                del out
    return t[1:].min(axis=0)


def test_first_evaluation_of_a_long_list(P, gpu_lib):
    t = evaluate(P, 5000, 6, 8)
    print("calls (ms):", *(f"{1e3 * x:.2f}" for x in t), flush=True)
    assert t[0] <= 1.45 * np.median(t[4:]) and t[1] <= 1.45 * np.median(t[4:])


def test_several_slices_cost_their_share(P, gpu_lib):
    one, three = evaluate(P, 100, 6, 8), evaluate(P, 300, 6, 8)
    print("1e5 pairs (us):", *(f"{1e6 * x:.0f}" for x in one), flush=True)
    print("3e5 pairs (us):", *(f"{1e6 * x:.0f}" for x in three), flush=True)
    assert np.median(three[4:]) <= 3.5 * np.median(one[4:])
