"""Transfers between the device and host memory of either kind: large pageable ones go through page-locked slots in
pieces, small hash batches through one page-locked buffer, batches of codes in chunks. Whatever the route, the bytes
are the same."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SLOT_COLUMNS = 16384  # columns of a 64-row tile that fills a slot of 4 MB


@pytest.mark.parametrize("K,N", [(1, 2), (64, 2 * SLOT_COLUMNS), (65, 2 * SLOT_COLUMNS + 2), (63, SLOT_COLUMNS - 2),
                                 (130, 5 * SLOT_COLUMNS + 6), (400, 2), (64, SLOT_COLUMNS), (64, SLOT_COLUMNS + 2),
                                 (2048, 512), (2047, 514), (400, 5242), (400, 5244)])
def test_matrices_through_the_slots(gpu, K, N):
    """Upload and download at tile edges (rows beside 64, columns beside a slot's), beside the largest matrix that goes
    in one piece (4 MB) and the smallest that goes up in tiles (8 MB), pageable and page-locked on either side."""
    from flyvec_amd import Hasher, Trainer, _lib
    W = np.random.default_rng(K).standard_normal((K, N), dtype=np.float32)
    locked = _lib.pinned_empty(W.shape, np.float32)
    locked[...] = W
    for source in (W, locked):
        t = Trainer(N // 2, K, 3, 16)
        t.set_weights(source)
        assert np.array_equal(t.get_weights().view(np.uint32), W.view(np.uint32))
        out = _lib.pinned_empty(W.shape, np.float32)
        assert np.array_equal(t.get_weights(out).view(np.uint32), W.view(np.uint32))
        t.close()
    if K > 1:
        h = Hasher(W)
        assert np.array_equal(h.weights(), W)
        h.close()
    assert _lib.load().fv_host_staging_release() == 0


@pytest.mark.parametrize("n", [1, (1 << 18) - 1, 1 << 18, (1 << 19) + 5, 5 * (1 << 17) - 1, 5 * (1 << 17),
                               (1 << 20) + 1, 3 * (1 << 20) - 1, 3 * (1 << 20), (1 << 22) + 3])
def test_orders_through_the_slots(gpu, n):
    """Window tables and orders of n 64-bit entries: beside the sizes from which pieces are taken (5 MB downwards, 24 MB
    upwards), whole and broken last pieces."""
    from flyvec_amd import Trainer
    rng = np.random.default_rng(n)
    tokens = rng.integers(0, 50, size=1000, dtype=np.int32)
    starts = rng.integers(0, 990, size=n).astype(np.uint64)
    perm = rng.permutation(n).astype(np.uint64)
    t = Trainer(50, 8, 5, 16)
    t.set_corpus_starts(tokens, starts)
    assert np.array_equal(t.window_starts(), starts)
    t.set_permutation(perm)
    assert np.array_equal(t.get_permutation(), perm)
    t.close()


def held():
    import ctypes as C
    from flyvec_amd import _lib
    out = C.c_size_t(0)
    _lib.check(_lib.load().fv_host_staging_held(C.byref(out)))
    return out.value


def test_what_transfers_page_lock(gpu):
    """Small and middling transfers page-lock one slot at most (a matrix of 3 MB took four, so did a corpus of 8 MB);
    large ones keep four for those that follow, until they are given back."""
    from flyvec_amd import Trainer, _lib
    slot = 4 << 20
    assert _lib.load().fv_host_staging_release() == 0 and held() == 0
    rng = np.random.default_rng(0)
    t = Trainer(50, 8, 5, 16)
    t.set_corpus_starts(rng.integers(0, 50, 2 << 20).astype(np.int32), rng.integers(0, 2 << 20, 600000).astype(np.uint64) // 2)
    t.set_permutation(rng.permutation(600000).astype(np.uint64))
    t.get_permutation()
    assert held() == 0
    t.close()
    t = Trainer(937, 400, 5, 16)
    W = rng.standard_normal((400, 2 * 937), dtype=np.float32)
    t.set_weights(W)
    assert held() == slot and np.array_equal(t.get_weights(), W) and held() == slot
    t.close()
    t = Trainer(4000, 400, 5, 16)
    W = rng.standard_normal((400, 2 * 4000), dtype=np.float32)
    t.set_weights(W)
    assert held() == 4 * slot and np.array_equal(t.get_weights(), W) and held() == 4 * slot
    t.close()
    assert _lib.load().fv_host_staging_release() == 0 and held() == 0


@pytest.mark.parametrize("n,slots", [(30000, 2), (60000, 4)])
def test_hash_batches_borrow_their_staging(gpu, n, slots):
    """Batches of codes for ordinary memory on one hasher after another page-lock two slots in all (four chunks of 1.7 MB) or
    four (of 3.2 MB); the results are the device-resident call's, on a hasher's first batch (one stream) and on later ones
    (two), and while other threads' transfers hold slots."""
    from flyvec_amd import Hasher, Trainer, _lib
    K = 400
    assert _lib.load().fv_host_staging_release() == 0
    rng = np.random.default_rng(5)
    W = rng.standard_normal((K, 200), dtype=np.float32)
    idx = rng.integers(0, 200, size=(n, 7)).astype(np.int32)
    want = None
    for i in range(3):
        h = Hasher(W)
        got = h.hash_windows(idx, 20, packed=False, codes=True)
        if want is None:
            dev, codes = _lib.DeviceBuffer.from_numpy(idx), _lib.DeviceBuffer(n * K)
            h.hash_windows_dev(dev, n, 7, 20, None, codes)
            h.sync()
            want = codes.to_numpy(np.int8, (n, K))
        assert np.array_equal(got, want) and held() == slots * (4 << 20)
        if i:
            assert np.array_equal(h.hash_windows(idx, 20, packed=False, codes=True), want) and held() == slots * (4 << 20)
        h.close()
    bad = []

    def matrices(seed):
        V = 40000
        M = np.random.default_rng(seed).standard_normal((130, 2 * V), dtype=np.float32)
        t = Trainer(V, 130, 3, 16)
        for _ in range(3):
            t.set_weights(M)
            if not np.array_equal(t.get_weights(), M):
                bad.append(seed)
        t.close()

    def hashes(seed):
        h = Hasher(W)
        for _ in range(6):
            if not np.array_equal(h.hash_windows(idx, 20, packed=False, codes=True), want):
                bad.append(seed)
        h.close()

    threads = [threading.Thread(target=matrices if s % 2 else hashes, args=(s,)) for s in range(6)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad


@pytest.mark.parametrize("slots", [0, 1, 3])
def test_every_route_with_fewer_slots_or_none(gpu, slots):
    """Where the process may page-lock nothing (as where the system gives nothing) every transfer goes the runtime's way,
    with one slot or three it waits for what there is: the same bytes. A limit below what is held gives back what is idle."""
    from flyvec_amd import Hasher, Trainer, _lib
    lib = _lib.load()
    slot = 4 << 20
    rng = np.random.default_rng(8)
    try:
        assert lib.fv_host_staging_limit(slots * slot + 5) == 0 and held() <= slots * slot
        for K, V in ((64, 500), (400, 1500), (130, 20000)):     # one piece; between; tiles
            W = rng.standard_normal((K, 2 * V), dtype=np.float32)
            t = Trainer(V, K, 3, 16)
            t.set_weights(W)
            assert np.array_equal(t.get_weights(), W)
            t.close()
        t = Trainer(50, 8, 5, 16)
        n = (1 << 22) + 3
        starts, perm = rng.integers(0, 990, size=n).astype(np.uint64), rng.permutation(n).astype(np.uint64)
        t.set_corpus_starts(rng.integers(0, 50, 1000).astype(np.int32), starts)
        t.set_permutation(perm)
        assert np.array_equal(t.window_starts(), starts) and np.array_equal(t.get_permutation(), perm)
        t.close()
        h = Hasher(rng.standard_normal((70, 400), dtype=np.float32))
        for n, w in ((30000, 3), (100003, 3), (140001, 11)):    # light indices twice, heavy ones on two streams
            idx = rng.integers(0, 400, size=(n, w)).astype(np.int32)
            dev, bits, codes = _lib.DeviceBuffer.from_numpy(idx), _lib.DeviceBuffer(n * 16), _lib.DeviceBuffer(n * 70)
            h.hash_windows_dev(dev, n, w, 9, bits, codes)
            h.sync()
            got = h.hash_windows(idx, 9, packed=True, codes=True)
            assert np.array_equal(got[0], bits.to_numpy(np.uint64, (n, 2))) and np.array_equal(got[1], codes.to_numpy(np.int8, (n, 70)))
            assert np.array_equal(h.hash_windows(idx, 9, packed=True), got[0])
        h.close()
        assert held() == slots * slot
    finally:
        assert lib.fv_host_staging_limit(1 << 40) == 0


def test_more_transfers_at_once_than_there_are_slots(gpu):
    """Six threads, each with a trainer of its own, hold up to four of eight slots each: they wait for each other's and
    all finish with their own matrix."""
    from flyvec_amd import Trainer
    K, V = 130, 30000
    bad = []

    def work(seed):
        W = np.random.default_rng(seed).standard_normal((K, 2 * V), dtype=np.float32)
        t = Trainer(V, K, 3, 16)
        for _ in range(3):
            t.set_weights(W)
            if not np.array_equal(t.get_weights(), W):
                bad.append(seed)
        t.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad


@pytest.mark.parametrize("K,w,n", [(400, 1, 1), (400, 1, 569), (400, 1, 570), (400, 1, 648), (400, 1, 649), (400, 1, 20000),
                                   (70, 11, 2016), (70, 11, 2017), (70, 11, 2299), (70, 11, 2300), (70, 11, 2301),
                                   (70, 11, 100003), (400, 11, 40001)])
@pytest.mark.parametrize("locked", [False, True])
def test_hash_batches_of_every_route(gpu, K, w, n, locked):
    """Codes and packed codes from host arrays, beside the largest batches that go through the one buffer (2^18 bytes of
    indices and codes: of one target with 400 neurons 569 with both kinds of code and 648 with plain codes only, of
    windows of 11 with 70 neurons 2016 and 2299), one chunk and several, against the device-resident call on the same
    indices. An index out of range is reported by every route and leaves the next call clean."""
    from flyvec_amd import Hasher, _lib
    V = 500
    rng = np.random.default_rng(n)
    h = Hasher(rng.standard_normal((K, 2 * V), dtype=np.float32))
    idx = rng.integers(-1, 2 * V, size=(n, w)).astype(np.int32)
    if w == 1:
        idx[:] = rng.integers(0, V, size=(n, 1))
    dev, bits_dev = _lib.DeviceBuffer.from_numpy(idx), _lib.DeviceBuffer(n * h.words * 8)
    codes_dev = _lib.DeviceBuffer(n * K)
    h.hash_windows_dev(dev, n, w, 9, bits_dev, codes_dev)
    h.sync()
    bits, codes = bits_dev.to_numpy(np.uint64, (n, h.words)), codes_dev.to_numpy(np.int8, (n, K))
    src = idx
    out = {}
    if locked:
        src = _lib.pinned_empty(idx.shape, np.int32)
        src[...] = idx
        out = dict(out_bits=_lib.pinned_empty(bits.shape, np.uint64), out_codes=_lib.pinned_empty(codes.shape, np.int8))
    for bad in (False, True, False):
        if bad:
            kept = src[n // 2, 0]
            src[n // 2, 0] = 2 * V
            with pytest.raises(_lib.FlyvecError):
                h.hash_windows(src, 9, packed=True, codes=True, **out)
            src[n // 2, 0] = kept
        else:
            got_bits, got_codes = h.hash_windows(src, 9, packed=True, codes=True, **out)
            assert np.array_equal(got_bits, bits) and np.array_equal(got_codes, codes)
    assert np.array_equal(h.hash_windows(src, 9, packed=False, codes=True), codes)
    if w == 1:
        idx += V  # the target block's columns
        dev2 = _lib.DeviceBuffer.from_numpy(idx)
        h.hash_windows_dev(dev2, n, 1, 9, None, codes_dev)
        h.sync()
        assert np.array_equal(h.hash_targets(idx[:, 0] - V, 9), codes_dev.to_numpy(np.int8, (n, K)))
    h.close()


def test_one_corpus_after_another(gpu, oracle_lib):
    """A trainer given corpora of other sizes in turn (a little smaller: the buffers are used again; much smaller, larger:
    they are not), with reshuffles between, samples what a new trainer would."""
    from flyvec_amd import Trainer
    from conftest import small_corpus
    V, w = 300, 7
    t = Trainer(V, 16, w, 64)
    for i, n in enumerate((20000, 19000, 4000, 4000, 60000, 55000)):
        tokens, offsets = small_corpus(n, V, seed=i)
        t.set_corpus(tokens, offsets)
        starts = oracle_lib.window_starts(offsets, w)
        assert t.num_windows == len(starts) and np.array_equal(t.window_starts(), starts)
        assert np.array_equal(t.get_permutation(), np.arange(len(starts), dtype=np.uint64))
        assert np.array_equal(t.inverse_frequency(), oracle_lib.inverse_frequency(tokens, V))
        t.shuffle(i)
        assert np.array_equal(np.sort(t.get_permutation()), np.arange(len(starts), dtype=np.uint64))
    with pytest.raises(Exception):
        t.set_corpus(np.full(100, V, dtype=np.int32), np.array([0, 50, 100], dtype=np.uint64))
    with pytest.raises(Exception):
        t.num_windows  # the corpus before the refused one is gone, as before
    t.close()


@pytest.mark.parametrize("n,nth", [(20000, 1), (20000, 2), (20000, 3), (20000, 4), (55000, 1)])
def test_a_corpus_that_fits_a_new_trainer_fits_one_that_has_a_corpus(gpu, oracle_lib, n, nth):
    """Where the device's memory does not hold what the call needs beside the buffers kept from the corpus before, they are
    given back and the corpus is set as on a new trainer: whichever allocation is refused (the second corpus much smaller, so
    that nothing is kept but while it fails, or a little, so that only the offsets' memory is new). On a new trainer the refusal
    stands, and the next corpus is set as ever."""
    from flyvec_amd import Trainer, _lib
    from conftest import small_corpus
    V, w = 300, 7
    big, tokens_offsets = small_corpus(60000, V, seed=1), small_corpus(n, V, seed=2)
    starts = oracle_lib.window_starts(tokens_offsets[1], w)

    def refuse(t):
        _lib.check(_lib.load().fv_trainer_fail_allocation(t.handle, nth))

    def check(t):
        assert np.array_equal(t.window_starts(), starts)
        assert np.array_equal(t.get_permutation(), np.arange(len(starts), dtype=np.uint64))
        assert np.array_equal(t.inverse_frequency(), oracle_lib.inverse_frequency(tokens_offsets[0], V))

    for given in (False, True):
        def set_corpus(t):
            if given:
                t.set_corpus_starts(tokens_offsets[0], starts)
            else:
                t.set_corpus(*tokens_offsets)
        t = Trainer(V, 16, w, 64)
        t.set_corpus(*big)
        t.shuffle(1)
        refuse(t)
        set_corpus(t)
        check(t)
        t.shuffle(2)
        assert np.array_equal(np.sort(t.get_permutation()), np.arange(len(starts), dtype=np.uint64))
        t.close()
        t = Trainer(V, 16, w, 64)
        refuse(t)
        with pytest.raises(_lib.FlyvecError) as e:
            set_corpus(t)
        assert e.value.code == _lib.FV_ERR_HIP and "allocation" in str(e.value)
        with pytest.raises(_lib.FlyvecError):
            t.num_windows
        set_corpus(t)
        check(t)
        t.close()
