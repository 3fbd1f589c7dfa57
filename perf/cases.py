"""The workloads this sampler's speed is measured on.

A case is one decode step: logits (or the hidden states in front of the output layer) of a
batch of requests, each with its own sampling settings, to one token per row.  Three calls
make such a step:

  sample   BatchedSampler.sample(), the serving engine's call: host lists in, host lists out
  launch   FusedSampler.launch(), the C ABI's fie_sampler_sample on resident arguments
  lmhead   FusedSampler.launch_lmhead(), the output layer and the sampler in one call
"""

from __future__ import annotations

import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "full-inference-engine_amd"))

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
LP_COLS = 20
# A request of the "sample" call ends after this many tokens; the next one takes its row.
REQUEST_TOKENS = 32


def listed():
    return [
        # One interactive user: the smallest step there is, latency and host work count.
        dict(name="sample_1_user", call="sample", rows=1, vocab=151936, dtype="bf16",
             logits="peaked", mix="nucleus", hist=0),
        # A batch that decodes greedily: one argmax per row, no sampling at all.
        dict(name="sample_64_greedy", call="sample", rows=64, vocab=151936, dtype="fp16",
             logits="peaked", mix="greedy", hist=0),
        # A loaded server's step as the engine makes it: every kind of request, penalties over
        # contexts that grow by a token a step, requests that end and are replaced.
        dict(name="sample_256_mixed", call="sample", rows=256, vocab=151936, dtype="fp16",
             logits="peaked", mix="mixed", hist=2048),
        # Few requests, half greedy and half at temperature 1 with no filter, in fp32.
        dict(name="step_8_plain", call="launch", rows=8, vocab=151936, dtype="fp32",
             logits="wide", mix="half_plain", hist=0),
        # Chat defaults: temperature, top-k and top-p together, no penalties.
        dict(name="step_64_topk", call="launch", rows=64, vocab=151936, dtype="fp32",
             logits="peaked", mix="topk_topp", hist=0),
        # The headline batch: greedy, top-k, top-p and both, all with penalties.
        dict(name="step_256_mixed", call="launch", rows=256, vocab=151936, dtype="fp16",
             logits="peaked", mix="mixed", hist=2048),
        # An API's open settings: high temperature, top-p near 1 or none, no top-k, so that
        # the nucleus runs thousands of tokens deep.
        dict(name="step_48_open", call="launch", rows=48, vocab=151936, dtype="bf16",
             logits="peaked", mix="open", hist=512),
        # An odd vocabulary (rows that are not 16-byte aligned), logprobs and min-p.
        dict(name="step_24_logprobs", call="launch", rows=24, vocab=50001, dtype="bf16",
             logits="peaked", mix="logprobs", hist=300),
        # The largest batch, on flat logits (an untrained or very hot model): every row's
        # nucleus holds most of the vocabulary.
        dict(name="step_1024_flat", call="launch", rows=1024, vocab=151936, dtype="bf16",
             logits="flat", mix="nucleus", hist=0),
        # A large vocabulary on a coarse grid (exact ties), top-k up to 1024, long contexts.
        dict(name="step_128_ties", call="launch", rows=128, vocab=262144, dtype="fp32",
             logits="ties", mix="wide_topk", hist=4096),
        # The output layer and the sampler together, a small decode batch: weights dominate.
        dict(name="lmhead_16", call="lmhead", rows=16, vocab=151936, dtype="bf16",
             logits="peaked", mix="mixed", hist=0, hidden=4096),
        # The same for a loaded server.
        dict(name="lmhead_256", call="lmhead", rows=256, vocab=151936, dtype="fp16",
             logits="peaked", mix="mixed", hist=512, hidden=4096),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over the logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    call = rng.choice(("sample", "launch", "launch", "launch", "lmhead"))
    rows = _spread(rng, 1, 256)
    vocab = _spread(rng, 4000, 262144)
    if rng.random() < 0.5:
        vocab -= vocab % 128                      # half of all models pad their vocabulary
    case = dict(call=call, rows=rows, vocab=vocab, dtype=rng.choice(tuple(DTYPES)),
                logits=rng.choice(("peaked", "peaked", "wide", "ties")))
    if call == "lmhead":
        case["dtype"] = rng.choice(("fp16", "bf16"))
        case["logits"] = "peaked"
        case["hidden"] = 128 * _spread(rng, 4, 32)
        case["vocab"] = min(vocab, 151936)
    if call == "launch" and rng.random() < 0.2:
        # flat logits: any number of rows up to the largest step's
        case["logits"], case["mix"] = "flat", "nucleus"
        case["rows"], case["vocab"] = _spread(rng, 8, 1024), min(vocab, 151936)
    else:
        mixes = ["half_plain", "topk_topp", "mixed", "nucleus", "wide_topk", "logprobs", "open"]
        case["mix"] = rng.choice(mixes + (["greedy"] if call == "sample" else []))
        if case["mix"] in ("half_plain", "logprobs", "open"):
            # few rows, as listed: such rows often need passes over all of their tokens
            case["rows"], case["vocab"] = min(rows, 48), min(vocab, 151936)
    case["hist"] = rng.choice((0, _spread(rng, 16, 4096))) if case["mix"] in PENALISED else 0
    return case


# ---------------------------------------------------------------------------- settings
PENALISED = ("mixed", "wide_topk", "open", "logprobs")


def _settings(case):
    """Each row's sampling settings, as keyword arguments."""
    rows, mix = case["rows"], case["mix"]
    got = []
    for i in range(rows):
        if mix == "greedy":
            p = {}
        elif mix == "half_plain":
            p = {} if i < rows // 2 else dict(temperature=1.0)
        elif mix == "topk_topp":
            p = dict(temperature=0.7, top_k=50, top_p=0.9)
        elif mix == "mixed":
            q, k, t = i * 4 // rows, (20, 50, 100)[i % 3], (0.8, 0.9, 0.95)[i % 3]
            p = dict(repetition_penalty=1.1, frequency_penalty=0.5, presence_penalty=0.3)
            if q:
                p["temperature"] = 0.7
            if q in (1, 3):
                p["top_k"] = k
            if q in (2, 3):
                p["top_p"] = t
        elif mix == "nucleus":
            p = dict(temperature=1.0 if case["logits"] == "flat" else 0.7, top_p=0.95)
        elif mix == "wide_topk":
            p = dict(temperature=1.0, top_k=(1, 64, 256, 1024)[i % 4], top_p=0.9,
                     repetition_penalty=1.2)
        elif mix == "logprobs":
            p = dict(temperature=(0.0, 0.6, 0.9)[i % 3], logprobs=(0, 5, 20, None)[i % 4])
            if i % 3 == 1:
                p["min_p"] = 0.05
            if i % 3 == 2:
                p["top_p"] = 0.9
            if i % 2:
                p["presence_penalty"] = 0.4
        elif mix == "open":
            p = dict(temperature=(0.8, 1.0, 1.2)[i % 3], top_p=(1.0, 0.95, 0.99, 1.0)[i % 4])
            if i % 2:
                p.update(presence_penalty=0.5, frequency_penalty=0.2)
        else:
            raise ValueError(mix)
        got.append(p)
    return got


# ---------------------------------------------------------------------------- inputs
def _logits(case, gen):
    """[rows, vocab] of the case's shape in its type.  peaked: a trained model's, about
    rank^-1.1 with noise; wide: N(0, 3); flat: N(0, 0.3); ties: N(0, 2) on the fp16 grid."""
    rows, vocab, kind = case["rows"], case["vocab"], case["logits"]
    x = torch.randn(rows, vocab, generator=gen, device=DEV)
    if kind == "peaked":
        ranks = torch.argsort(torch.rand(rows, vocab, generator=gen, device=DEV), dim=1)
        x = 0.5 * x - 1.1 * torch.log(ranks.float() + 1.0)
    elif kind == "wide":
        x = 3.0 * x
    elif kind == "flat":
        x = 0.3 * x
    elif kind == "ties":
        x = (2.0 * x).half().float()
    return x.to(DTYPES[case["dtype"]])


def _head(case, gen):
    """(hidden, weight) whose product has the peaked shape: one shared direction carries
    the ranks, the rest is noise."""
    rows, vocab, H, dt = case["rows"], case["vocab"], case["hidden"], DTYPES[case["dtype"]]
    d = torch.randn(H, generator=gen, device=DEV)
    d /= d.norm()
    hidden = d + 0.01 * torch.randn(rows, H, generator=gen, device=DEV) / H ** 0.5
    ranks = torch.randperm(vocab, generator=gen, device=DEV).float()
    weight = 0.5 * torch.randn(vocab, H, generator=gen, device=DEV)
    weight += (-1.1 * torch.log(ranks + 1.0))[:, None] * d
    return hidden.to(dt), weight.to(dt)


def _contexts(case, rng):
    """Each row's context: `hist` ids, Zipf(1.1) over a shuffled vocabulary, without id 0;
    None where the case keeps no contexts."""
    if not case["hist"]:
        return None
    vocab = case["vocab"]
    p = np.cumsum(np.arange(1, vocab, dtype=np.float64) ** -1.1)
    ids = 1 + rng.permutation(vocab - 1)
    at = np.searchsorted(p, rng.random((case["rows"], case["hist"])) * p[-1])
    return [row.tolist() for row in ids[np.minimum(at, vocab - 2)]]


def _inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = _head(case, gen) if case["call"] == "lmhead" else _logits(case, gen)
    return x, _contexts(case, np.random.default_rng(seed))


# ---------------------------------------------------------------------------- the calls
def prepare(case, seed):
    from fie_amd.batching.sampler import SHARED_STREAM, BatchedSampler, resolve_params
    from fie_amd.kernel import FusedSampler
    from fie_amd.runtime.sampling import SamplingParams

    x, contexts = _inputs(case, seed)
    params = [SamplingParams(**p) for p in _settings(case)]
    state = dict(call=case["call"], x=x, params=params)
    rows = case["rows"]
    if case["call"] == "sample":
        state.update(sampler=BatchedSampler(DEV, generator_seed=seed), prompts=contexts,
                     contexts=None if contexts is None else [list(c) for c in contexts],
                     ids=list(range(rows)), steps=0)
        return state
    rng = np.empty((rows, 3), dtype=np.uint64)
    rng[:, 0], rng[:, 1], rng[:, 2] = seed, SHARED_STREAM, np.arange(rows)
    hp = resolve_params(params, case["vocab"], None, contexts, rng=rng)
    fs = FusedSampler(DEV)
    buf = fs.step_buffers(rows, hp.tail_ints())
    buf.dev.zero_()
    buf.stage(hp)
    buf.upload(torch.cuda.current_stream())
    logits = x
    if case["call"] == "lmhead":
        logits = torch.zeros(rows, case["vocab"], dtype=DTYPES[case["dtype"]], device=DEV)
        state.update(hidden=x[0], weight=x[1])
    fs.ensure_workspace(rows, case["vocab"])
    state.update(fs=fs, buf=buf, logits=logits, args=fs.build_args(logits, buf, hp),
                 out=_outputs(buf, case, logits))
    return state


def _outputs(buf, case, logits):
    """The step's results, as the device arrays that the call fills."""
    rows = case["rows"]

    def at(name, dtype, width=1):
        o = buf.offs[name]
        t = buf.dev[o:o + rows * width * torch.empty(0, dtype=dtype).element_size()].view(dtype)
        return t.view(rows, width) if width > 1 else t

    out = dict(tokens=at("tokens", torch.int64))
    if case["call"] == "lmhead":
        out["logits"] = logits
        return out
    out.update(row_max=at("row_max", torch.float32), top_k_key=at("tk_key", torch.int32),
               cut=at("cut_comp", torch.int64), kept_mass=at("kept_mass", torch.int64, 2))
    if case["mix"] == "logprobs":
        out.update(chosen_logprob=at("chosen_lp", torch.float32),
                   top_ids=at("top_ids", torch.int64, LP_COLS),
                   top_logprobs=at("top_lp", torch.float32, LP_COLS))
    return out


def run(state):
    if state["call"] == "launch":
        state["fs"].launch(state["args"])
        return state["out"]
    if state["call"] == "lmhead":
        state["fs"].launch_lmhead(state["args"], state["hidden"], state["weight"])
        return state["out"]
    sampler, contexts, ids = state["sampler"], state["contexts"], state["ids"]
    if state["steps"] == REQUEST_TOKENS:          # the requests have ended: new ones take their rows
        state["steps"] = 0
        sampler.forget(ids)
        ids = state["ids"] = [i + len(ids) for i in ids]
        if contexts is not None:
            contexts = state["contexts"] = [list(c) for c in state["prompts"]]
    result = sampler.sample(state["x"], state["params"], contexts, ids)
    state["steps"] += 1
    if contexts is not None:
        for context, token in zip(contexts, result.token_ids):
            context.append(token)
    out = dict(tokens=np.array(result.token_ids))
    if result.logprobs:
        entries = [e for row in sorted(result.logprobs) for e in result.logprobs[row]]
        out.update(ids=np.array([e[0] for e in entries]),
                   logprobs=np.array([e[1] for e in entries], dtype=np.float32))
    return out


# ---------------------------------------------------------------------------- what it takes
def work(case):
    rows, vocab = case["rows"], case["vocab"]
    size = 4 if case["dtype"] == "fp32" else 2
    moved = rows * vocab * size + 4 * rows * case["hist"] + 48 * rows
    flops = 2 * rows * vocab
    if case["call"] == "lmhead":
        moved += (rows + vocab) * case["hidden"] * size
        flops += 2 * rows * vocab * case["hidden"]
    return dict(bytes=moved, flops=flops)


def tolerance(case):
    """Tokens, cuts, thresholds and masses are whole numbers of exact rules and stay the
    same.  Floats: fp32 roundings of fp64 logprobs and the fp32 row maximum; for the output
    layer, fp32 sums rounded to the logits' type, where another order of the sum moves a
    value by one unit of that type now and then."""
    if case["call"] == "lmhead":
        # four times what a library product on the same operands differs by
        return (dict(rel=2.5e-5, max=1e-3, differ=0.01) if case["dtype"] == "fp16"
                else dict(rel=1.6e-4, max=8e-3, differ=0.01))
    return dict(rel=3e-7, max=1e-6)


def _fp32(v):
    """A setting as the call takes it, an fp32 value."""
    return float(np.float32(v))


def exact(case, seed):
    """The floating outputs in 64 bits: row maxima and best logprobs of the penalised,
    scaled logits, or the output layer's logits.  The draw has no such value."""
    if case["call"] == "sample":
        return None
    x, contexts = _inputs(case, seed)
    if case["call"] == "lmhead":
        hidden, weight = x[0].double(), x[1]
        cuts = range(0, weight.shape[0], 16384)
        logits = torch.cat([hidden @ weight[i:i + 16384].double().T for i in cuts], dim=1)
        return dict(tokens=None, logits=logits)
    settings = _settings(case)
    y = x.double()
    if contexts is not None:
        for r, p in enumerate(settings):
            ids, n = np.unique(contexts[r], return_counts=True)
            at = torch.from_numpy(ids).to(DEV)
            v, rep = y[r, at], _fp32(p.get("repetition_penalty", 1.0))
            v = torch.where(v > 0, v / rep, v * rep) - _fp32(p.get("presence_penalty", 0.0))
            y[r, at] = v - _fp32(p.get("frequency_penalty", 0.0)) * torch.from_numpy(n).to(DEV).double()
    # greedy rows (temperature 0, or top-k 1) are not scaled
    scale = [_fp32(p.get("temperature", 0.0)) if p.get("top_k", 0) != 1 else 0.0 for p in settings]
    y /= torch.tensor([t or 1.0 for t in scale], device=DEV, dtype=torch.float64)[:, None]
    out = dict(tokens=None, row_max=y.max(dim=1).values, top_k_key=None, cut=None, kept_mass=None)
    if case["mix"] == "logprobs":
        best = torch.zeros(case["rows"], LP_COLS, dtype=torch.float64, device=DEV)
        for r, p in enumerate(settings):
            n = p["logprobs"] or 0
            best[r, :n] = torch.log_softmax(y[r], 0).topk(n).values
        out.update(chosen_logprob=None, top_ids=None, top_logprobs=best)
    return out
