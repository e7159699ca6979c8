"""The dense launch that visits only the rows of the matrix somebody needs (fv_train_rows.h), against the checker."""
import numpy as np
import pytest

from conftest import small_corpus

pytestmark = pytest.mark.gpu


def _trainer(tokens, offsets, V, K, w, B, W0, delta=0.0, lr0=1e-3, mode=2, **kw):
    from flyvec_amd import Trainer
    t = Trainer(V, K, w, B, initial_learning_rate=lr0, delta=delta, **kw)
    t.set_row_updates(mode)
    t.set_corpus(tokens, offsets)
    perm = np.random.default_rng(6).permutation(t.num_windows).astype(np.uint64)
    t.set_permutation(perm)
    t.set_weights(W0)
    return t, perm


@pytest.mark.parametrize("V,K,w,B,n_tokens,delta", [
    (3000, 100, 7, 40, 12000, 0.0),      # few rows touched: most lag until they are 16 steps behind
    (3000, 100, 7, 40, 12000, 0.4),
    (500, 400, 11, 512, 60000, 0.0),     # nearly every row touched in every step
    (700, 209, 5, 333, 40000, 0.3),
    (300, 1, 3, 7, 2000, 0.0),           # one neuron, one group of which three parts are padding
    (200, 5, 1, 3, 900, 0.0),            # window of one position
    (90, 2048, 7, 64, 6000, 0.0),        # the widest rows: xx kept for 8 steps, two threads per group of a round
    (2000, 1025, 4, 100, 20000, 0.0),
    (40000, 64, 5, 500, 60000, 0.0),     # more rounds of rows than a thread has groups in flight in the launch over all rows
    (1500, 8, 6, 20000, 90000, 0.0),     # grouped by a launch of its own
    (4100, 513, 6, 2000, 60000, 0.0),
])
def test_epochs_with_rows_updated_as_they_are_needed(gpu, oracle_lib, V, K, w, B, n_tokens, delta):
    """Two epochs (partial last minibatch included) against the checker's, the log line's norms in between."""
    from flyvec_amd import synthetic
    to = oracle_lib
    tokens, offsets = small_corpus(n_tokens, V, seed=K)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = synthetic.synapses(K, V, seed=3, sigma=0.02)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0, delta=delta)
    Wo = W0.copy()
    n_steps = (len(starts) + B - 1) // B
    for ep in (3, 4):
        norms = t.row_norms(K)
        assert np.allclose(norms, np.sqrt((Wo.astype(np.float64) ** 2).sum(1)), rtol=1e-12)
        t.run_epoch(ep, 15)
        wo = to.train_steps(Wo, tokens, starts, perm, 0, B, n_steps, w, invf, to.epoch_eps(1e-3, ep, 15),
                            delta=t.epoch_delta(ep, 15))
        last = len(starts) - (n_steps - 1) * B
        assert np.array_equal(t.winners(last), wo[-last:])
        assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32)), ep
    assert t.row_update_steps >= 2 * n_steps - 1      # the first step on a new matrix visits every row
    assert sum(t.dense_path_counts) == 2 * n_steps and t.giveups_recovered == 0
    t.close()


def _planted(tokens, V, K):
    """Weights whose largest entries sit on the most frequent tokens: the dense term decides max|ds|."""
    from flyvec_amd import synthetic
    W = synthetic.synapses(K, V, seed=9)
    W[:, np.argsort(-np.bincount(tokens[tokens >= 0], minlength=V))[:3]] = np.float32(7.0)
    return W


@pytest.mark.parametrize("delta", [0.0, 0.3])
@pytest.mark.parametrize("wait", [None, 0])
def test_the_maximum_is_not_the_sparse_elements(gpu, oracle_lib, wait, delta):
    """The launch then goes over every row twice, with an exchange between its blocks; where that gives up (a limit of zero
    rounds: every block decides at once) run_epoch takes up again with the separate launches, and rows that lacked
    updates have them."""
    to = oracle_lib
    V, K, w, B = 3000, 96, 9, 200
    tokens, offsets = small_corpus(40000, V, seed=2)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = _planted(tokens, V, K)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0, delta=delta)
    Wo = W0.copy()
    steps = 25
    eps = 1e-3
    for s in range(steps):
        if s == 10 and wait is not None:
            break
        t.step(s * B, B, eps, delta)
    done = s if wait is not None and s == 10 else steps
    to.train_steps(Wo, tokens, starts, perm, 0, B, done, w, invf, eps, delta=delta)
    assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32))
    known, made = t.dense_path_counts
    assert t.row_update_steps >= done - 1 and made >= 3
    if wait is not None:
        t._set_wait_limit(wait)
        t.run_epoch(3, 15)
        n_steps = (len(starts) + B - 1) // B
        to.train_steps(Wo, tokens, starts, perm, 0, B, n_steps, w, invf, to.epoch_eps(1e-3, 3, 15), delta=t.epoch_delta(3, 15))
        assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32))
        assert t.giveups_recovered == 1 and t.dense_launches == 2
    t.close()


@pytest.mark.parametrize("launches", [0, 1, 2])
@pytest.mark.parametrize("drained", [False, True])
def test_dense_launches_chosen_behind_a_launch_that_gave_up(gpu, oracle_lib, launches, drained):
    """A launch that visits rows gives up (a limit of zero rounds), steps are enqueued behind it, more of them than steps
    whose xx is kept, and the form of the dense launches is chosen anew before anybody has heard of it (drained: behind a
    call that waits and does not report it, and more steps in front of the report). The matrix stays as the last step in
    front of that launch left it, the report says so, and steps go on from there."""
    from flyvec_amd._lib import FlyvecError
    to = oracle_lib
    V, K, w, B = 3000, 96, 9, 200
    tokens, offsets = small_corpus(40000, V, seed=2)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = _planted(tokens, V, K)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0)
    eps, live, behind = 1e-3, 10, 25
    for s in range(live):
        t.step(s * B, B, eps)
    t.sync()
    t._set_wait_limit(0)
    for s in range(live, live + behind):
        t.step(s * B, B, eps)
    assert t.row_update_steps >= live + behind - 2
    if drained:
        t.winners(B)
    t.set_dense_launches(launches)
    t._set_wait_limit(1 << 14)

    def six_steps(W):
        to.train_steps(W, tokens, starts, perm, 40 * B, B, 6, w, invf, eps)
        return W

    if drained:
        for s in range(40, 46):
            t.step(s * B, B, eps)
    with pytest.raises(FlyvecError, match="gave up"):
        t.sync()
    W = t.get_weights()
    Wo, at = W0.copy(), None
    for s in range(live + behind):
        if s >= live and np.array_equal(W.view(np.uint32), (six_steps(Wo.copy()) if drained else Wo).view(np.uint32)):
            at = s
            break
        to.train_steps(Wo, tokens, starts, perm, s * B, B, 1, w, invf, eps)
    assert at is not None and at < live + behind - 17
    if not drained:
        for s in range(40, 46):
            t.step(s * B, B, eps)
        assert np.array_equal(t.get_weights().view(np.uint32), six_steps(Wo).view(np.uint32))
    t.close()


@pytest.mark.parametrize("synapses", ["small", "middling", "planted"])
def test_chosen_by_the_sizes_and_by_what_the_launches_find(gpu, oracle_lib, synapses):
    """Three epochs of 253 steps, the form chosen as by default. The largest |ds| of the sparse elements is 40 to 115 times
    the dense ones' bound (small: the form is taken but for the first steps on a new matrix, through several refreshes of
    the bound), 1.4 to 3.8 times (middling: it is entered and left, as a launch that finds less than twice ends it), or just the
    largest of all (planted: no launch finds it clear and the form is never taken)."""
    from flyvec_amd import synthetic
    to = oracle_lib
    V, K, w, B = 12000, 100, 5, 200
    tokens, offsets = small_corpus(60000, V, seed=2)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = _planted(tokens, V, K) if synapses == "planted" else synthetic.synapses(K, V, seed=3, sigma=0.02 if synapses == "small" else 0.11)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0, lr0=5e-4, mode=0)
    Wo = W0.copy()
    n_steps = (len(starts) + B - 1) // B
    for ep in (3, 4, 5):
        t.run_epoch(ep, 15)
        to.train_steps(Wo, tokens, starts, perm, 0, B, n_steps, w, invf, to.epoch_eps(5e-4, ep, 15))
        assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32)), ep
    taken, known = t.row_update_steps, t.dense_path_counts[0]
    assert n_steps == 254 and sum(t.dense_path_counts) == 3 * n_steps
    if synapses == "small":
        assert taken >= 3 * n_steps - 10 and known >= 3 * n_steps - 1
    elif synapses == "middling":
        assert 0 < taken < 3 * n_steps - 100
    else:
        assert taken == 0
    t.close()


@pytest.mark.parametrize("eps,taken", [(6.2e-4, True), (6.3e-4, False)])
def test_left_alone_beyond_the_largest_learning_rate(gpu, oracle_lib, eps, taken):
    """The bound of |W| grows by |eps| a step: by the sizes the form asks for 32 steps between two refreshes of it."""
    from flyvec_amd import synthetic
    to = oracle_lib
    V, K, w, B, n_steps = 12000, 100, 5, 200, 40
    tokens, offsets = small_corpus(60000, V, seed=2)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = synthetic.synapses(K, V, seed=3, sigma=0.02)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0, mode=0)
    for rep in range(2):  # (the first steps' answers are in hand)
        for s in range(rep * n_steps, (rep + 1) * n_steps):
            t.step(s * B, B, eps)
        t.sync()
    Wo = W0.copy()
    to.train_steps(Wo, tokens, starts, perm, 0, B, 2 * n_steps, w, invf, np.float32(eps))
    assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32))
    assert t.row_update_steps >= n_steps - 9 if taken else t.row_update_steps == 0
    t.close()


@pytest.mark.parametrize("order", ["short", "strided", "again", "six and a jump", "twelve and a jump"])
def test_steps_that_do_not_follow_each_other(gpu, oracle_lib, order):
    """Steps on windows that are not the ones behind the last step's: a sequence per step would settle the whole matrix
    every time, so by the sizes the form is not taken; from eight steps in order on it is."""
    from flyvec_amd import synthetic
    to = oracle_lib
    V, K, w, B, n_steps, eps = 12000, 210, 5, 200, 60, 2e-4
    tokens, offsets = small_corpus(60000, V, seed=2)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = synthetic.synapses(K, V, seed=3, sigma=0.02)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0, mode=0)
    N = len(starts) // B
    run = {"six and a jump": 6, "twelve and a jump": 12}.get(order, 1)
    at = [(s % N if order == "short" else 3 * s % N if order == "strided" else 4 if order == "again" else
           (s // run * 31 + s % run) % (N - 1)) * B for s in range(n_steps)]
    n = B - 7 if order == "short" else B
    Wo = W0.copy()
    for s in range(12):
        t.step(s * B, B, eps)
        to.train_steps(Wo, tokens, starts, perm, s * B, B, 1, w, invf, eps)
    t.sync()
    before = t.row_update_steps
    for first in at:
        t.step(first, n, eps)
        to.train_step(Wo, to.inflate(tokens, starts, perm, first, n, w, V), invf, eps)
    taken = t.row_update_steps - before
    assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32))
    assert taken >= n_steps - 12 if run == 12 else taken == 0
    t.close()


@pytest.mark.parametrize("mode", [0, 2])
def test_steps_are_enqueued_without_waiting_for_the_device(gpu, mode):
    """2000 steps of 30 to 40 us: the host is done with them long before the device is (8 to 10 us a step)."""
    import time
    from flyvec_amd import synthetic
    V, K, w, B, n_steps = 20000, 400, 11, 4000, 2000
    tokens, offsets = small_corpus(1500000, V, seed=2)
    t, _ = _trainer(tokens, offsets, V, K, w, B, synthetic.synapses(K, V, seed=3, sigma=0.02), mode=mode)
    N = t.num_windows // B
    t.step(0, B, 2e-4)
    t.sync()
    before, ratios = t.row_update_steps, []
    for _ in range(3):
        t0 = time.perf_counter()
        for s in range(n_steps):
            t.step(s % N * B, B, 2e-4)
        t1 = time.perf_counter()
        t.sync()
        ratios.append((t1 - t0) / (time.perf_counter() - t0))
    assert t.row_update_steps - before > n_steps / 4
    assert min(ratios) < 0.6, ratios
    t.close()


@pytest.mark.parametrize("entries", [1, 3])
def test_more_sentinels_than_a_wave_notes(gpu, oracle_lib, entries):
    from flyvec_amd import synthetic
    to = oracle_lib
    V, K, w, B = 700, 130, 9, 900
    tokens, offsets = small_corpus(40000, V, seed=8)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = synthetic.synapses(K, V, seed=2, sigma=0.02)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0)
    t.set_sentinel_list(entries)
    Wo = W0.copy()
    n_steps = (len(starts) + B - 1) // B
    t.run_epoch(3, 15)
    to.train_steps(Wo, tokens, starts, perm, 0, B, n_steps, w, invf, to.epoch_eps(1e-3, 3, 15))
    assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32)) and t.row_update_steps >= n_steps - 1
    t.close()


def test_calls_between_steps_see_every_update(gpu, oracle_lib):
    """Steps that visit rows, broken off in every way a caller can: look at the matrix, replace it, another order, another
    place in it, another size of minibatch, another trainer's steps beside them, the separate launches."""
    from flyvec_amd import Trainer, synthetic
    to = oracle_lib
    V, K, w, B = 2500, 61, 6, 150
    tokens, offsets = small_corpus(30000, V, seed=5)
    starts, invf = to.window_starts(offsets, w), to.inverse_frequency(tokens, V)
    W0 = synthetic.synapses(K, V, seed=3, sigma=0.02)
    t, perm = _trainer(tokens, offsets, V, K, w, B, W0)
    other = Trainer(V, 8, w, 16)
    other.set_corpus(tokens, offsets)
    other.set_weights(synthetic.synapses(8, V, seed=1))
    Wo = W0.copy()

    def steps(first, n, count):
        for s in range(count):
            t.step(first + s * n, n, 1e-3)
            to.train_step(Wo, to.inflate(tokens, starts, perm, first + s * n, n, w, V), invf, 1e-3)

    def same(what):
        assert np.array_equal(t.get_weights().view(np.uint32), Wo.view(np.uint32)), what

    steps(0, B, 20)
    assert np.allclose(t.row_norms(K), np.sqrt((Wo.astype(np.float64) ** 2).sum(1)), rtol=1e-12)
    steps(20 * B, B, 7)
    same("steps behind the norms")
    steps(27 * B, B, 5)
    Wo = synthetic.synapses(K, V, seed=4, sigma=0.02)
    t.set_weights(Wo)
    steps(32 * B, B, 9)
    perm = np.random.default_rng(7).permutation(len(starts)).astype(np.uint64)
    t.set_permutation(perm)
    steps(0, B, 6)
    t.shuffle(3)
    perm = t.get_permutation()
    steps(0, B, 6)
    steps(50 * B + 3, B, 6)
    steps(10 * B + 1, B - 7, 6)
    same("another order, place and size")
    steps(0, B, 6)
    other.step(0, 16, 1e-4)
    steps(6 * B, B, 4)
    other.sync()
    steps(10 * B, B, 4)
    same("another trainer in flight")
    steps(0, B, 6)
    before = t.row_update_steps
    t.set_dense_launches(2)
    steps(6 * B, B, 3)
    t.set_dense_launches(0)
    steps(9 * B, B, 5)
    xx, nc = t.step_stats()
    ref = to.train_step(Wo.copy(), to.inflate(tokens, starts, perm, 0, B, w, V), invf, 1e-3)
    steps(0, B, 1)
    xx, nc = t.step_stats()
    assert np.array_equal(xx, ref["xx"]) and nc == ref["nc"]
    same("separate launches")
    assert t.row_update_steps > before > 30
    t.set_row_updates(1)
    steps(0, B, 3)
    same("every row")
    assert t.time_steps(0, 20, 1e-3, per_kernel=False)[0] > 0 and t.time_steps_graph(0, 4, 1e-3, 2) > 0
    t.close()
    other.close()
