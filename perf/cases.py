"""The sampling path's workloads, for timing and for comparing two builds.

A case is a dict of plain values naming one call of the package's public entry
points at one size: a sampling step (SamplerContext.sample), a row's kept
distribution (SamplerContext.distribution), the logits producers (lm_head,
lm_head_q8) and the JSON-object mask producers (json_mask, JsonMaskSet.fill).
`listed()` holds the twelve cases that stand for the path's use, `draw(rng)`
one more of the same ranges.  Inputs are synthetic and made on the GPU from the
seed; their shapes and distributions are those of the benchmark's
configurations (tachyon_amd/workloads.py, bench.py).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from tachyon_amd import constrain, device, lmhead
from tachyon_amd import workloads as wl

QWEN = wl.QWEN_VOCAB      # 151936
LLAMA = wl.LLAMA_VOCAB    # 128256


# ---- the cases -----------------------------------------------------------------

def _sample(**kw):
    """A sampling step: `rows` rows of `usable` ids (`stride` apart) with one set of settings for every row, or the
    four kinds of the mixed batch."""
    c = dict(kind="sample", rows=1, usable=QWEN, stride=0, sigma=3.0, spikes=0, temperature=0.7, top_k=0, top_p=1.0,
             min_p=0.0, repetition=1.0, presence=0.0, frequency=0.0, history=0, zipf=False, mask="none", n_logprobs=0,
             mixed=False)
    c.update(kw)
    c["stride"] = c["stride"] or c["usable"]
    return c


def listed():
    return [
        # one sequence decoding: the smallest call, where launches and latency count
        _sample(name="sample_b1", rows=1, spikes=20, top_k=40, top_p=0.9, repetition=1.1, history=64),
        # a small server's step: every request with its own settings (greedy, plain temperature, top-k + top-p, min-p)
        _sample(name="sample_mixed_b32", rows=32, sigma=2.0, temperature=1.0, presence=0.5, frequency=0.3,
                history=512, zipf=True, mixed=True),
        # a full batch with every feature on: all penalties over long histories, a mask, top-k, top-p, min-p, logprobs
        _sample(name="sample_full_b256", rows=256, temperature=0.7, top_k=64, top_p=0.92, min_p=0.02, repetition=1.1,
                presence=0.4, frequency=0.2, history=1024, zipf=True, mask="third", n_logprobs=5),
        # the largest batch, no top-k and flat logits: the nucleus spans most of the vocabulary
        _sample(name="sample_nucleus_b1024", rows=1024, sigma=1.0, temperature=1.2, top_p=0.98, repetition=1.05,
                history=256),
        # speculative decoding: the target's kept distributions of a drafted run, at the reference's default settings
        dict(_sample(rows=8, temperature=0.7, top_k=20, top_p=0.8, repetition=1.05, history=64), name="distribution_b8",
             kind="distribution", dist_stride=20),
        # the output layer of one decoding sequence: the weights' one read
        dict(name="lm_head_b1", kind="lm_head", rows=1, dim=4096, vocab=QWEN, split=True),
        # ... of a small batch, activations rounded to bf16
        dict(name="lm_head_bf16_b48", kind="lm_head", rows=48, dim=4096, vocab=QWEN, split=False),
        # ... of a full batch (or a prompt's rows when every position's logits are wanted)
        dict(name="lm_head_b256", kind="lm_head", rows=256, dim=4096, vocab=QWEN, split=True),
        # the quantized output layer of a few decoding sequences, and of a full batch
        dict(name="lm_head_q8_b4", kind="lm_head_q8", rows=4, dim=4096, vocab=QWEN),
        dict(name="lm_head_q8_b256", kind="lm_head_q8", rows=256, dim=4096, vocab=QWEN),
        # response_format json_object: the masks of a full batch, each row in a state of its own document, and a step
        # of a serving loop that keeps recent states' masks
        dict(name="json_mask_b256", kind="json_mask", rows=256, vocab=QWEN, usable=QWEN),
        dict(name="json_fill_b256", kind="json_fill", rows=256, vocab=QWEN, usable=QWEN),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["sample"] * 5 + ["distribution", "lm_head", "lm_head", "lm_head_q8", "lm_head_q8", "json_mask",
                                        "json_fill"])
    if kind in ("sample", "distribution"):
        usable = rng.choice([QWEN, LLAMA, 151669, 32000, _log_int(rng, 3000, QWEN)])
        way = rng.choice(["topk", "masked", "full", "nucleus", "minp", "mixed"]) if kind == "sample" else \
            rng.choice(["topk", "nucleus"])
        history = _log_int(rng, 16, 1024) if rng.random() < 0.7 else 0
        c = _sample(rows=_log_int(rng, 1, 256), usable=usable, stride=usable + rng.choice([0, 0, 1, 3, 64]),
                    sigma=rng.choice([1.0, 2.0, 3.0]), temperature=rng.choice([0.5, 0.7, 0.8, 1.0, 1.2]),
                    history=history, zipf=rng.random() < 0.5, repetition=1.1 if history and rng.random() < 0.7 else 1.0)
        if way in ("topk", "masked", "full"):
            c.update(top_k=rng.choice([20, 40, 50, 64, _log_int(rng, 1, 200)]), top_p=rng.choice([0.8, 0.9, 0.95, 1.0]))
        if way in ("masked", "full"):
            c.update(mask=rng.choice(["grammar", "third"]), n_logprobs=rng.choice([0, 5, 20]))
        if way == "full" and history:
            c.update(presence=0.4, frequency=0.2, min_p=0.02)
        if way == "nucleus":
            c.update(top_p=rng.choice([0.8, 0.9, 0.95, 0.98, 1.0]), rows=_log_int(rng, 1, 768))
        if way == "minp":
            c.update(min_p=rng.choice([0.02, 0.05, 0.1]))
        if way == "mixed":
            c.update(mixed=True, temperature=1.0, presence=0.5 if history else 0.0, rows=max(4, c["rows"] // 4))
        if kind == "distribution":
            c.update(kind=kind, rows=_log_int(rng, 2, 16), dist_stride=c["top_k"] or 1024)
        return c
    if kind in ("lm_head", "lm_head_q8"):
        dim = rng.choice([1024, 2048, 3584, 4096, 5120, 64 * rng.randint(8, 80)])
        vocab = min(rng.choice([QWEN, LLAMA, 32000, _log_int(rng, 3000, QWEN)]), 4096 * QWEN // dim)
        c = dict(kind=kind, rows=_log_int(rng, 1, 256), dim=dim, vocab=vocab)
        if kind == "lm_head":
            c["split"] = rng.random() < 0.6
        return c
    vocab = rng.choice([QWEN, LLAMA, 32000, _log_int(rng, 3000, QWEN)])
    return dict(kind=kind, rows=_log_int(rng, 1, 256), vocab=vocab, usable=vocab - rng.choice([0, 0, 13]))


# ---- inputs --------------------------------------------------------------------

def _generator(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _params(case):
    rows = case["rows"]
    p = wl.make_params(rows, temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"],
                       repetition_penalty=case["repetition"], presence_penalty=case["presence"],
                       frequency_penalty=case["frequency"], min_p=case["min_p"],
                       flags=(wl.ROW_CONSTRAINED if case["mask"] != "none" else 0)
                       | (wl.ROW_LOGPROBS if case["n_logprobs"] else 0), n_logprobs=case["n_logprobs"])
    if case["mixed"]:
        q = rows // 4
        p["temperature"][:q] = 0.0
        p["top_k"][2 * q:3 * q] = 50
        p["top_p"][2 * q:3 * q] = 0.95
        p["min_p"][3 * q:] = 0.05
    return p


def _histories(case, rng):
    if not case["history"]:
        return None, None
    make = wl.zipf_histories if case["zipf"] else wl.uniform_histories
    return make(rng, case["rows"], case["history"], case["usable"])


def _logits(case, seed):
    gen = _generator(seed, 1)
    x = torch.randn(case["rows"], case["stride"], generator=gen, device="cuda") * case["sigma"]
    if case["spikes"]:
        at = torch.randint(0, case["usable"], (case["rows"], case["spikes"]), generator=gen, device="cuda")
        x.scatter_add_(1, at, torch.full(at.shape, 8.0, device="cuda"))
    return x


def _allowed(case, seed, rng):
    """bool [rows, usable]: 30% of the ids, or per row a share log-uniform in [0.1%, 60%], in ranges (even rows) or
    scattered (odd rows)."""
    rows, n = case["rows"], case["usable"]
    at = torch.rand(rows, n, generator=_generator(seed, 2), device="cuda")
    if case["mask"] == "third":
        return at < 0.3
    share = np.exp(rng.uniform(math.log(0.001), math.log(0.6), rows))
    allowed = at < torch.from_numpy(share.astype(np.float32)).cuda()[:, None]
    for r in range(0, rows, 2):
        allowed[r] = False
        runs = int(rng.integers(1, 9))
        for length in rng.multinomial(max(1, int(share[r] * n)), np.ones(runs) / runs):
            s = int(rng.integers(0, n - int(length) + 1))
            allowed[r, s:s + int(length)] = True
    return allowed


def _pack(allowed):
    rows, n = allowed.shape
    words = (n + 31) // 32
    bits = torch.nn.functional.pad(allowed, (0, words * 32 - n)).view(rows, words, 32).to(torch.int32)
    out = torch.zeros(rows, words, dtype=torch.int32, device="cuda")
    for b in range(32):
        out |= bits[:, :, b] << b
    return out


def _sampling_inputs(case, seed):
    """Everything of a sampling call: the logits and the mask's bits on the GPU, the rest on the host."""
    rng = np.random.default_rng(int(seed))
    ids, offsets = _histories(case, rng)
    allowed = None if case["mask"] == "none" else _allowed(case, seed, rng)
    return dict(logits=_logits(case, seed), params=_params(case), ids=ids, offsets=offsets, allowed=allowed,
                uniforms=wl.uniforms(rng, case["rows"]))


def _sampling_state(case, seed):
    n = _sampling_inputs(case, seed)
    rows = case["rows"]
    # the row kinds come from what the host knows of the step: settings and history lengths
    host = wl.Workload("", np.empty((rows, 0), np.float32), case["usable"], n["params"], n["ids"], n["offsets"], None,
                       n["uniforms"])
    batch = device.DeviceBatch(
        logits=n["logits"], usable=case["usable"], params=torch.from_numpy(n["params"].view(np.uint8)).cuda(),
        hist_ids=None if n["ids"] is None else torch.from_numpy(n["ids"].view(np.int32)).cuda(),
        hist_offsets=None if n["offsets"] is None else torch.from_numpy(n["offsets"].view(np.int32)).cuda(),
        mask=None if n["allowed"] is None else _pack(n["allowed"]), uniforms=torch.from_numpy(n["uniforms"]).cuda(),
        top_stride=max(1, case["n_logprobs"]), row_kinds=device.row_kinds(host, n["allowed"] is not None),
        dist_kinds=device.row_kinds(host, False))
    return batch


@functools.lru_cache(maxsize=4)
def _vocabulary(n):
    """The tokenizer: one per vocabulary size, whatever the step's inputs."""
    tokens, special = wl.json_vocab(n)
    return constrain.HostVocab.from_tokens(tokens, special)


def _constraint(prefix):
    c = constrain.JsonConstraint()
    c.advance(prefix)
    return c


FILL_STEPS = 64  # steps of the decoding loop that json_fill runs through
FILL_KEPT = 1024  # states whose masks the set keeps


def _documents(case, seed):
    """json_fill: per step, the rows' prefixes; each row writes documents of its own, a 4-byte token a step."""
    rng = np.random.default_rng(int(seed))
    steps = [[] for _ in range(FILL_STEPS)]
    for _ in range(case["rows"]):
        doc = wl.json_document(rng)
        at = int(rng.integers(0, len(doc) + 1))
        for s in steps:
            if at >= len(doc):
                doc, at = wl.json_document(rng), 0
            s.append(doc[:at])
            at += 4
    return steps


def prepare(case, seed):
    k = case["kind"]
    if k in ("sample", "distribution"):
        s = dict(case=case, batch=_sampling_state(case, seed), ctx=device.SamplerContext(case["rows"], case["usable"]))
        if k == "sample":
            s["out"] = device.Outputs(case["rows"], max(1, case["n_logprobs"]))
        return s
    if k in ("lm_head", "lm_head_q8"):
        rows, dim, vocab = case["rows"], case["dim"], case["vocab"]
        gen = _generator(seed, 3)
        s = dict(case=case, x=torch.randn(rows, dim, generator=gen, device="cuda") * 3.0,
                 g=1.0 + 0.2 * torch.randn(dim, generator=gen, device="cuda"),
                 out=torch.empty(rows, vocab, dtype=torch.float32, device="cuda"))
        if k == "lm_head":
            s["w"] = torch.empty(vocab, dim, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=gen)
            s["ws"] = torch.empty(lmhead.workspace_bytes(rows, dim, case["split"]), dtype=torch.uint8, device="cuda")
        else:
            s["w"] = torch.randint(-127, 128, (vocab, dim), generator=gen, device="cuda", dtype=torch.int8)
            s["wscale"] = (0.001 * torch.randn(vocab, dim // 32, generator=gen, device="cuda")).half().view(torch.int16)
            s["ws"] = torch.empty(lmhead.workspace_bytes_q8(rows, dim), dtype=torch.uint8, device="cuda")
        return s
    vocab = constrain.DeviceVocab(_vocabulary(case["vocab"]))
    stride = (case["usable"] + 31) // 32
    mask = torch.zeros(case["rows"], stride, dtype=torch.int32, device="cuda")
    s = dict(case=case, vocab=vocab, mask=mask, stride=stride, step=0)
    if k == "json_mask":
        packed = constrain.pack_states([_constraint(p) for p in wl.json_prefixes(case["rows"], seed=int(seed))])
        s["states"] = torch.from_numpy(packed).cuda()
    else:
        s["set"] = constrain.JsonMaskSet(case["rows"], FILL_KEPT, case["usable"])
        s["steps"] = [constrain.JsonMaskSet.pack([_constraint(p) for p in prefixes])
                      for prefixes in _documents(case, seed)]
    return s


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "sample":
        o = state["out"]
        state["ctx"].sample(state["batch"], o, with_logprobs=case["n_logprobs"] > 0)
        got = dict(token=o.token, prob=o.prob, keep=o.keep)
        if case["n_logprobs"]:
            got.update(logprob=o.logprob, top_ids=o.top_ids, top_lp=o.top_lp)
        return got
    if k == "distribution":
        ids, probs, keep = state["ctx"].distribution(state["batch"], case["dist_stride"])
        return dict(ids=ids, probs=probs, keep=keep)
    if k == "lm_head":
        return lmhead.lm_head(state["x"], state["g"], 1e-6, state["w"], split=case["split"], out=state["out"],
                              workspace=state["ws"])
    if k == "lm_head_q8":
        return lmhead.lm_head_q8(state["x"], state["g"], 1e-6, state["w"], state["wscale"], out=state["out"],
                                 workspace=state["ws"])
    if k == "json_mask":
        constrain.json_mask(state["vocab"], state["states"], case["rows"], case["usable"], state["mask"],
                            state["stride"])
        return state["mask"]
    state["set"].fill(state["vocab"], state["steps"][state["step"] % FILL_STEPS], state["mask"], state["stride"])
    state["step"] += 1
    return state["mask"]


# ---- what a pass cannot do without, and what its results may differ by ----------

def work(case):
    k, rows = case["kind"], case["rows"]
    if k in ("sample", "distribution"):
        n = case["usable"]
        b = rows * (4 * n + 4 * case["history"] + 4 + 40 + 12)
        if case["mask"] != "none":
            b += rows * 4 * ((n + 31) // 32)
        if case["n_logprobs"]:
            b += rows * (4 + 8 * case["n_logprobs"])
        if k == "distribution":
            b += rows * 8 * case["dist_stride"]
        return dict(bytes=b, flops=0)
    if k in ("lm_head", "lm_head_q8"):
        dim, vocab = case["dim"], case["vocab"]
        weights = vocab * dim * 2 if k == "lm_head" else vocab * (dim + dim // 32 * 2)
        # split activations are two bf16 values, each multiplied with the weights
        products = rows * vocab * dim * (2 if case.get("split") else 1)
        return dict(bytes=weights + rows * dim * 4 + dim * 4 + rows * vocab * 4, flops=2 * products)
    # the masks written, and the states; the vocabulary's bytes once where a mask has to be evaluated
    v = _vocabulary(case["vocab"])
    b = rows * (12 + 4 * ((case["usable"] + 31) // 32))
    return dict(bytes=b + v.bytes.nbytes + v.offsets.nbytes + v.special.nbytes, flops=0)


def tolerance(case):
    k = case["kind"]
    if k in ("sample", "distribution"):
        # tokens, kept counts and ids are the same; f32 sums of up to 151936 exponentials in another order, and the
        # logarithm of one
        return dict(rel=1e-6, max=4e-6, differ=0.0)
    if k == "lm_head":
        # hi + lo holds an activation to 2^-17 of itself; one bf16 value to 2^-9
        return dict(rel=1e-5, max=1e-4) if case["split"] else dict(rel=7e-3, max=6e-2)
    return "exact"  # the quantized head's sums have a fixed order; masks are bits


# ---- the results in 64 bits ------------------------------------------------------

def _norm64(case, s):
    x, g = s["x"].double(), s["g"].double()
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-6) * g


def _exact_lm(case, seed):
    s = prepare(case, seed)
    xb = _norm64(case, s)
    out = torch.empty(case["rows"], case["vocab"], dtype=torch.float64, device="cuda")
    if case["kind"] == "lm_head_q8":
        nb = case["dim"] // 32
        blocks = xb.view(case["rows"], nb, 32)
        d = blocks.abs().amax(dim=2, keepdim=True) / 127.0
        q = blocks / d
        xb = (torch.sign(q) * torch.floor(q.abs() + 0.5) * d).reshape(case["rows"], case["dim"])
    for v in range(0, case["vocab"], 16384):
        w = s["w"][v:v + 16384].double()
        if case["kind"] == "lm_head_q8":
            w = w.view(w.shape[0], nb, 32) * s["wscale"][v:v + 16384].view(torch.float16).double()[:, :, None]
            w = w.reshape(w.shape[0], case["dim"])
        out[:, v:v + 16384] = xb @ w.t()
    return out


def _exact_distribution(case, seed):
    """The kept probabilities, best first: penalties, top-k, softmax, top-p, each row normalised over what is kept."""
    n = _sampling_inputs(case, seed)
    rows, usable, stride = case["rows"], case["usable"], case["dist_stride"]
    out = torch.zeros(rows, stride, dtype=torch.float64, device="cuda")
    for r in range(rows):
        y = n["logits"][r, :usable].double()
        if n["ids"] is not None:
            ids, counts = np.unique(n["ids"][n["offsets"][r]:n["offsets"][r + 1]], return_counts=True)
            at = torch.from_numpy(ids.astype(np.int64)).cuda()
            v = y[at]
            rep = float(np.float32(case["repetition"]))
            v = torch.where(v > 0, v / rep, v * rep) - case["presence"]
            y[at] = v - case["frequency"] * torch.from_numpy(counts.astype(np.float64)).cuda()
        y = torch.sort(y, descending=True).values
        t = float(np.float32(case["temperature"]))
        y = y[:case["top_k"]] if case["top_k"] else y[y >= y[0] - 30.0 * t]
        p = torch.exp((y - y[0]) / t)
        if case["top_p"] < 1.0:
            before = torch.cumsum(p, 0) / p.sum()
            p = p[:int((before < float(np.float32(case["top_p"]))).sum()) + 1]
        p = p / p.sum()
        m = min(stride, p.numel())
        out[r, :m] = p[:m]
    return dict(ids=None, probs=out, keep=None)


def exact(case, seed):
    k = case["kind"]
    if k in ("lm_head", "lm_head_q8"):
        return _exact_lm(case, seed)
    if k == "distribution":
        return _exact_distribution(case, seed)
    if k == "sample" and case["n_logprobs"]:
        # the alternatives; the pick and its probability hang on where the draw falls between two kept ids
        x = _logits(case, seed)[:, :case["usable"]]
        top = torch.topk(x, case["n_logprobs"], dim=1).values.double()
        lse = torch.stack([torch.logsumexp(row.double(), 0) for row in x])
        return dict(token=None, prob=None, keep=None, logprob=None, top_ids=None, top_lp=top - lse[:, None])
    return None
