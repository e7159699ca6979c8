"""Grouping by winner in a launch of its own: minibatches around 16384 and 65536 windows, one, two and four neurons a block."""
import numpy as np
import pytest

from conftest import small_corpus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [16384, 16385, 32768, 40001, 65535, 65536, 65537])
@pytest.mark.parametrize("heavy", [False, True])
def test_minibatches_at_the_edges_of_the_grouping_forms(gpu, oracle_lib, B, heavy):
    """Two whole minibatches, then a short one, then a whole one with the anti-Hebbian term and one without; with and
    without a neuron that wins most windows, so that a thread has more matches than it fetches ahead."""
    _steps(oracle_lib, B, heavy, 9)


@pytest.mark.parametrize("K", [256, 257, 512, 513, 518, 2047])
@pytest.mark.parametrize("heavy", [False, True])
def test_several_neurons_a_block(gpu, oracle_lib, K, heavy):
    """The same at the numbers of neurons where a block takes one more (the last block with fewer than that)."""
    _steps(oracle_lib, 17003, heavy, K)


def _steps(to, B, heavy, K):
    from flyvec_amd import Trainer, synthetic
    V, w = 300, 3
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


def test_a_neuron_that_wins_everything_does_not_hold_up_the_launch(gpu):
    """50000 windows of one neuron: 55 to 65 us on an otherwise idle device (a serial path through them took 480)."""
    from flyvec_amd import Trainer, synthetic
    for K in (64, 400, 1000):
        V, w, B = 2000, 3, 50000
        tokens, offsets = small_corpus(200000, V, seed=1, mean_chunk=40)
        W0 = synthetic.synapses(K, V, seed=3, sigma=0.02)
        W0[4] += 1.0
        t = Trainer(V, K, w, B)
        t.set_corpus(tokens, offsets)
        t.set_weights(W0)
        t.step(0, B, 1e-9)
        assert np.all(t.winners(B) == 4)
        assert min(t._time_kernel(1, 10) for _ in range(3)) < 0.2, K
        t.close()
