"""The work users have this package do, as cases for measurement: hashing of words and context windows, loading a
model, setting up a corpus, and training epochs, through the public Python classes.

Sizes: the command line's defaults (K = 400, w = 11, B = 10000), the benchmark's headline and large configurations
(V = 20000 and V = 50000, K = 1000, w = 15, B = 50000), the small models of the tests, and ragged sizes between.
Token ids follow a Zipf law over the vocabulary, windows carry their centre in the target block, some positions are
masked, synapses are normal: what the benchmark and the tests use.
"""
import ctypes
import math

import numpy as np
import torch

from flyvec_amd import _lib
from flyvec_amd.engine import Hasher, Trainer

LEARNING_RATE = 2.0e-4
N_EPOCHS = 15
PREC = 1.0e-30
DELTA = 0.4


def listed():
    return [
        # the codes of a sentence's tokens: one small call, host arrays in and out
        dict(name="sentence", kind="targets", K=400, V=20000, n=24, k=50, zipf=1.07),
        # the codes of a whole vocabulary in one call (simple_word_vectors, the per-word code table)
        dict(name="vocabulary", kind="targets", K=400, V=20000, n=20000, k=50, zipf=0.0),
        # a corpus shard of context windows, resident on the device, packed codes: the benchmark's hash workload
        dict(name="windows_packed", kind="windows_dev", K=400, V=20000, w=11, n=1 << 20, k=32, zipf=1.07, masked=0.0, packed=True),
        # the benchmark's large model, one code per byte, stop words masked
        dict(name="windows_K1000", kind="windows_dev", K=1000, V=50000, w=15, n=65537, k=50, zipf=1.0, masked=0.1, packed=False),
        # a batch of context windows between ordinary host arrays (get_context_embeddings)
        dict(name="windows_host", kind="windows_host", K=400, V=20000, w=11, n=100003, k=50, zipf=1.07, masked=0.1, packed=False),
        # a checkpoint taken into service: upload, normalisation, the matrix read back and a first batch of codes
        dict(name="load_model", kind="load", K=400, V=20000, k=50, n=64),
        # a corpus handed to a trainer: upload, 1/frequency, window table, shuffle
        dict(name="corpus", kind="corpus", V=20000, w=11, tokens=4_000_001, chunk=25, zipf=1.07),
        # an epoch of the command line's default model with its log line and its checkpoint; a partial last batch
        dict(name="epoch", kind="epoch", K=400, V=20000, w=11, B=10000, windows=1_003_217, chunk=25, zipf=1.07, delta=0.0),
        # the same model with the anti-Hebbian term
        dict(name="epoch_delta", kind="epoch", K=400, V=20000, w=11, B=10000, windows=403_217, chunk=25, zipf=1.07, delta=DELTA),
        # the benchmark's large model
        dict(name="epoch_large", kind="epoch", K=1000, V=50000, w=15, B=50000, windows=2_000_003, chunk=40, zipf=1.0, delta=0.0),
        # a model of odd sizes between the two
        dict(name="epoch_ragged", kind="epoch", K=209, V=7919, w=7, B=3001, windows=301_313, chunk=25, zipf=1.07, delta=0.0),
        # one minibatch of a model as small as the tests use: launches and latency
        dict(name="epoch_small", kind="epoch", K=64, V=1009, w=5, B=512, windows=512, chunk=25, zipf=1.07, delta=0.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["targets", "windows_dev", "windows_dev", "windows_host", "load", "corpus", "epoch", "epoch", "epoch", "epoch"])
    K, V = _log_int(rng, 50, 1000), _log_int(rng, 1000, 50000)
    w = rng.randint(3, 15)
    zipf = round(rng.uniform(0.9, 1.1), 3)
    chunk = rng.choice([25, 40])
    k = max(1, min(rng.choice([16, 32, 50]), K // 4))
    if kind == "targets":
        return dict(kind=kind, K=K, V=V, n=_log_int(rng, 1, 20000), k=k, zipf=zipf)
    if kind in ("windows_dev", "windows_host"):
        most = min(1 << 20, int(4.0e9 / (w * K))) if kind == "windows_dev" else 200000
        return dict(kind=kind, K=K, V=V, w=w, n=_log_int(rng, 100, most), k=k, zipf=zipf,
                    masked=rng.choice([0.0, 0.1]), packed=rng.random() < 0.5)
    if kind == "load":
        return dict(kind=kind, K=min(K, 400), V=min(V, 20000), k=min(k, 50), n=rng.randint(1, 200))
    if kind == "corpus":
        return dict(kind=kind, V=V, w=w, tokens=_log_int(rng, 20000, 4_000_000), chunk=chunk, zipf=zipf)
    B = _log_int(rng, 300, 50000)
    return dict(kind=kind, K=K, V=V, w=w, B=B, windows=_log_int(rng, B, max(B + 1, min(1_000_000, 60 * B))), chunk=chunk,
                zipf=zipf, delta=rng.choice([0.0, 0.0, 0.0, DELTA]))


# ---- inputs ------------------------------------------------------------------------------------------------------

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed, part):
    g = torch.Generator(device=_device())
    g.manual_seed(1000 * int(seed) + part)
    return g


def _ids(n, V, zipf, gen):
    """n token ids in [1, V), P(id = r) proportional to r^-zipf (id 0 is <UNK>)."""
    p = torch.arange(1, V, dtype=torch.float64, device=_device()) ** (-zipf)
    cdf = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(n, dtype=torch.float64, device=_device(), generator=gen)
    return (1 + torch.searchsorted(cdf, u, right=True)).clamp_(max=V - 1).to(torch.int32)


def _synapses(K, V, sigma, seed):
    return torch.randn(K, 2 * V, device=_device(), generator=_generator(seed, 1)).mul_(sigma)


def _corpus(case, n_tokens, seed):
    """About n_tokens token ids and the chunks' offsets on the host: the lengths are the quantiles of a geometric
    distribution in an order of the seed's own (so every seed has as many tokens and windows)."""
    gen = _generator(seed, 2)
    chunks = max(1, int(n_tokens / case["chunk"]))
    u = (torch.randperm(chunks, device=_device(), generator=gen).double() + 0.5) / chunks
    lengths = (torch.log1p(-u) / math.log1p(-1.0 / case["chunk"])).ceil_().clamp_(min=1).to(torch.int64)
    offsets = np.concatenate([[0], torch.cumsum(lengths, 0).cpu().numpy()]).astype(np.uint64)
    return _ids(int(offsets[-1]), case["V"], case["zipf"], gen).cpu().numpy(), offsets


def _windows(case, seed):
    """(n, w) column indices: context ids, the centre shifted into the target block, -1 = masked."""
    gen = _generator(seed, 3)
    n, w = case["n"], case["w"]
    idx = _ids(n * w, case["V"], case["zipf"], gen).view(n, w)
    idx[:, w // 2] += case["V"]
    if case["masked"]:
        idx[torch.rand(n, w, device=_device(), generator=gen) < case["masked"]] = -1
    return idx


def _target_ids(case, seed):
    if case["zipf"] == 0.0:
        return torch.randperm(case["V"], device=_device(), generator=_generator(seed, 4))[:case["n"]].to(torch.int32)
    return _ids(case["n"], case["V"], case["zipf"], _generator(seed, 4))


def _window_starts(offsets, w):
    """Corpus position of every window of chunks of w .. 213 tokens, in order."""
    start = offsets[:-1].astype(np.int64)
    length = offsets[1:].astype(np.int64) - start
    keep = (length >= w) & (length < 214)
    start, count = start[keep], length[keep] - w + 1
    first = np.cumsum(count) - count
    return np.repeat(start - first, count) + np.arange(int(count.sum()), dtype=np.int64)


def _epoch_inputs(case, seed):
    """Tokens, offsets, the windows' starts and their order: exactly case["windows"] windows, the epoch's."""
    per_token = math.exp(-case["w"] / case["chunk"])  # windows per token of geometric chunks
    tokens, offsets = _corpus(case, int(case["windows"] / per_token * 1.15) + 20 * case["chunk"] * case["w"], seed)
    starts = _window_starts(offsets, case["w"])[:case["windows"]]
    assert len(starts) == case["windows"]
    order = torch.randperm(len(starts), device=_device(), generator=_generator(seed, 5)).cpu().numpy()
    return tokens, starts, order


class _Resident:
    """A torch tensor as the device buffer the *_dev calls take."""

    def __init__(self, tensor):
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "targets":
        return dict(kind=kind, k=case["k"], ids=_target_ids(case, seed).cpu().numpy(),
                    hasher=Hasher(_synapses(case["K"], case["V"], 1.0, seed).cpu().numpy()))
    if kind in ("windows_dev", "windows_host"):
        hasher = Hasher(_synapses(case["K"], case["V"], 1.0, seed).cpu().numpy())
        idx = _windows(case, seed)
        if kind == "windows_host":
            return dict(kind=kind, k=case["k"], packed=case["packed"], hasher=hasher, idx=idx.cpu().numpy())
        idx = idx.contiguous()
        out = torch.zeros(case["n"], hasher.words, dtype=torch.int64, device=_device()) if case["packed"] else \
            torch.zeros(case["n"], case["K"], dtype=torch.int8, device=_device())
        torch.cuda.synchronize()
        return dict(kind=kind, k=case["k"], packed=case["packed"], hasher=hasher, idx=idx, idx_buf=_Resident(idx),
                    out=out, out_buf=_Resident(out))
    if kind == "load":
        return dict(kind=kind, k=case["k"], W=_synapses(case["K"], case["V"], 0.02, seed).cpu().numpy(),
                    ids=_ids(case["n"], case["V"], 1.07, _generator(seed, 4)).cpu().numpy())
    if kind == "corpus":
        tokens, offsets = _corpus(case, case["tokens"], seed)
        return dict(kind=kind, tokens=tokens, offsets=offsets, seed=seed, trainer=Trainer(case["V"], hid=64, window=case["w"], batch=512))
    tokens, starts, order = _epoch_inputs(case, seed)
    trainer = Trainer(case["V"], hid=case["K"], window=case["w"], batch=case["B"], initial_learning_rate=LEARNING_RATE,
                      delta=case["delta"], prec=PREC)
    trainer.set_corpus_starts(tokens, starts)
    trainer.set_permutation(order)
    trainer.set_weights(_synapses(case["K"], case["V"], 0.02, seed).cpu().numpy())
    # the page-locked array that checkpoints are taken through
    return dict(kind=kind, trainer=trainer, checkpoint=_lib.pinned_empty((case["K"], 2 * case["V"]), np.float32))


def run(state):
    kind = state["kind"]
    if kind == "targets":
        return state["hasher"].hash_targets(state["ids"], state["k"])
    if kind == "windows_dev":
        n, w = state["idx"].shape
        bits, codes = (state["out_buf"], None) if state["packed"] else (None, state["out_buf"])
        state["hasher"].hash_windows_dev(state["idx_buf"], n, w, state["k"], bits, codes)
        return state["out"]
    if kind == "windows_host":
        out = state["hasher"].hash_windows(state["idx"], state["k"], packed=state["packed"], codes=not state["packed"])
        return out.view(np.int64) if state["packed"] else out
    if kind == "load":
        hasher = Hasher(state["W"])
        hasher.normalize()
        out = dict(codes=hasher.hash_targets(state["ids"], state["k"]), synapses=hasher.weights())
        hasher.close()
        return out
    if kind == "corpus":
        t = state["trainer"]
        t.set_corpus(state["tokens"], state["offsets"])
        t.shuffle(state["seed"])
        return dict(windows=t.num_windows, inverse_frequency=t.inverse_frequency(), order=t.get_permutation().view(np.int64))
    t = state["trainer"]
    norms = t.row_norms(10)
    t.run_epoch(N_EPOCHS // 2, N_EPOCHS)
    return dict(norms=norms, synapses=t.get_weights(state["checkpoint"]))


# ---- what a pass needs, and what it gives ------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "corpus":  # tokens read; 1/frequency and the order of the windows written, the latter about one a token
        n_windows = case["tokens"] * math.exp(-case["w"] / case["chunk"])
        return dict(bytes=4 * case["tokens"] + 4 * case["V"] + 8 * n_windows, flops=case["tokens"])
    K, N = case["K"], 2 * case["V"]
    if kind == "targets":
        return dict(bytes=4 * K * min(case["n"], case["V"]) + 4 * case["n"] + K * case["n"], flops=K * case["n"])
    if kind in ("windows_dev", "windows_host"):
        n, w = case["n"], case["w"]
        out = 8 * ((K + 63) // 64) if case["packed"] else K
        return dict(bytes=4 * K * min(N, n * w) + 4 * n * w + out * n, flops=(w + 1) * K * n)
    if kind == "load":  # the matrix in and out, and read for the norms and read and written for the division
        return dict(bytes=20 * K * N + 5 * K * case["n"], flops=3 * K * N)
    # a step reads and writes the matrix and visits every window position's element and 1/frequency
    steps = -(-case["windows"] // case["B"])
    positions = case["windows"] * case["w"]
    return dict(bytes=8 * K * N * steps + 16 * positions + 4 * K * N, flops=positions * K + 3 * K * N * steps)


def tolerance(case):
    if case["kind"] in ("epoch", "load"):
        return dict(rel=1.0e-6)  # measured against exact: 2.5e-7
    if case["kind"] == "corpus":
        return dict(rel=1.2e-7)  # 2.8e-8
    return "exact"


def _codes(act, k):
    """act > mean of the k-th and (k+1)-th largest, by row."""
    top = torch.topk(act, k + 1, dim=1).values
    return act > (top[:, k - 1:k] + top[:, k:k + 1]) / 2


def _pack(code):
    n, K = code.shape
    words = (K + 63) // 64
    full = torch.zeros(n, words * 64, dtype=torch.int64, device=code.device)
    full[:, :K] = code
    return (full.view(n, words, 64) << torch.arange(64, device=code.device)).sum(2)


def _window_activations(Wt, idx):
    """Sum of the window's rows of Wt (token-major, a zero row last), in float64."""
    idx = torch.where(idx < 0, Wt.shape[0] - 1, idx.to(torch.int64))
    act = torch.zeros(idx.shape[0], Wt.shape[1], dtype=torch.float64, device=Wt.device)
    for c in range(idx.shape[1]):
        act += Wt[idx[:, c]]
    return act


def _with_zero_row(W):
    return torch.cat([W.t().double(), torch.zeros(1, W.shape[0], dtype=torch.float64, device=W.device)])


def _exact_epoch(case, seed):
    K, V, w, B = case["K"], case["V"], case["w"], case["B"]
    tokens, starts, order = _epoch_inputs(case, seed)
    tok = torch.from_numpy(tokens).to(_device()).to(torch.int64)
    starts = torch.from_numpy(starts[order]).to(_device())
    count = torch.bincount(tok, minlength=V).clamp(max=1 << 24).double()
    invf = torch.where(count > 0, 1.0 / count, 0.0)
    W = _synapses(K, V, 0.02, seed).t().double().contiguous()
    norms = W[:, :10].square().sum(0).sqrt()
    epoch = N_EPOCHS // 2
    eps = LEARNING_RATE * (1.0 - epoch / N_EPOCHS)
    delta = case["delta"] * 0.5 * (1.0 + math.tanh((epoch - 0.125 * N_EPOCHS) / 10.0))
    column = torch.arange(w, device=_device()) == w // 2
    for first in range(0, case["windows"], B):
        s = starts[first:first + B]
        t = tok[s[:, None] + torch.arange(w, device=_device())]
        idx, f = t + V * column, invf[t]
        act = _window_activations(W, idx)  # no position is masked
        best = act.topk(2 if delta else 1, dim=1).indices
        xx = torch.zeros(K, dtype=torch.float64, device=_device())
        sparse = torch.zeros(2 * V * K, dtype=torch.float64, device=_device())
        for rank, strength in ((0, 1.0), (1, -delta)):
            if strength == 0.0:
                continue
            win = best[:, rank]
            xx.index_add_(0, win, strength * (W[idx, win[:, None]] * f).sum(1))
            sparse.index_add_(0, (idx * K + win[:, None]).view(-1), (strength * f).view(-1))
        ds = sparse.view(2 * V, K).addcmul_(W, xx, value=-1.0)
        step = ds.mul_(eps / max(PREC, max(float(ds.max()), -float(ds.min()))))
        W += torch.where(step.abs() > 1e-10, step, 0.0)
    return dict(norms=norms, synapses=W.t().contiguous())


def exact(case, seed):
    kind = case["kind"]
    if kind == "corpus":
        tokens, offsets = _corpus(case, case["tokens"], seed)
        count = np.bincount(tokens, minlength=case["V"]).astype(np.float64)
        invf = np.divide(1.0, count, out=np.zeros_like(count), where=count > 0)
        return dict(windows=len(_window_starts(offsets, case["w"])), inverse_frequency=invf, order=None)
    if kind == "epoch":
        return _exact_epoch(case, seed)
    W = _synapses(case["K"], case["V"], 0.02 if kind == "load" else 1.0, seed)
    if kind == "load":
        W = W.double()
        W /= W.square().sum(1, keepdim=True).sqrt() + 1e-32
        ids = _ids(case["n"], case["V"], 1.07, _generator(seed, 4)).to(torch.int64)
        return dict(codes=_codes(W[:, case["V"] + ids].t(), case["k"]).to(torch.int8), synapses=W)
    Wt = _with_zero_row(W)
    if kind == "targets":
        return _codes(Wt[case["V"] + _target_ids(case, seed).to(torch.int64)], case["k"]).to(torch.int8)
    idx, out = _windows(case, seed), []
    for part in idx.split(32768):
        code = _codes(_window_activations(Wt, part), case["k"])
        out.append(_pack(code) if case["packed"] else code.to(torch.int8))
    return torch.cat(out)
