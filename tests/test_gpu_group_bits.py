"""Grouping by winner from the rows of winner bits, in a launch of its own (minibatches of 16385 to 65536 windows)."""
import numpy as np
import pytest

from conftest import small_corpus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [16384, 16385, 32768, 40001, 65535, 65536, 65537])
@pytest.mark.parametrize("heavy", [False, True])
def test_minibatches_at_the_edges_of_the_grouping_forms(gpu, oracle_lib, B, heavy):
    """Two whole minibatches, then a short one (rows of bits that a longer minibatch filled are clear again), then a whole one
    with the anti-Hebbian term (grouped from the winner arrays) and one without; with and without a neuron that wins
    most windows, so that a thread has more matches than it fetches ahead."""
    from flyvec_amd import Trainer, synthetic
    to = oracle_lib
    V, K, w = 300, 9, 3
    tokens, offsets = small_corpus(200000, V, seed=1, mean_chunk=40)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = synthetic.synapses(K, V, seed=3, sigma=0.02)
    if heavy:
        W0[4] += 0.03
    t = Trainer(V, K, w, B, initial_learning_rate=1e-3)
    t.set_corpus(tokens, offsets)
    perm = np.random.default_rng(6).permutation(t.num_windows).astype(np.uint64)
    t.set_permutation(perm)
    t.set_weights(W0)
    Wo = W0.copy()
    for first, n, delta in ((0, B, 0.0), (B, B, 0.0), (7, 130, 0.0), (11, B, 0.3), (5, B, 0.0)):
        t.step(first, n, 1e-3, delta)
        ref = to.train_step(Wo, to.inflate(tokens, starts, perm, first, n, w, V), invf, 1e-3, delta=delta)
        xx, nc = t.step_stats()
        assert np.array_equal(t.winners(n), ref["winners"]) and np.array_equal(xx, ref["xx"]) and nc == ref["nc"], (first, n, delta)
    assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32))
    t.close()
