"""The calls whose speed counts, over the sizes they are used at.

Each case is one pass through the package's public entry points (or two, where
a program makes them one after the other): the sampler over rows of logits,
the softmax family, the output projection.  Inputs are made on the GPU from a
seed; the parameters of the sampling recipes are those of the benchmark's
workloads.  The families:

  chat       one blocking Sampler.sample + accept on a host row of logits: the
             drop-in for a program whose model runs on the CPU
  decode     one token's tail: output projection of the hidden states, then
             generate_step on its logits (chat loops, one or several contexts)
  generate   generate_step over the rows of several contexts' logits
  penalties  sample, top-k, frequency / presence penalties and logit biases
  zipf       sample, full sort with top-p and min-p over a peaked row
  topk       sample, a plain top-k of any size over a flat row
  mixed      sample, rows of unlike parameters (greedy, min-p, top-k, top-p)
             and many exactly equal values
  toptokens  top_tokens_device: the n most probable ids of every row
  softmax    softmax_device of every row
  logprob    log_prob_device of every row (scoring a continuation)
  perplexity the output projection of a chunk of positions, then row_nll_device
  head       the output projection alone
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch


def _package():
    """The package of the working folder (its folder's name is no identifier)."""
    if "nimllm_amd" not in sys.modules:
        root = os.path.join(os.getcwd(), "nim.llm_amd")
        spec = importlib.util.spec_from_file_location(
            "nimllm_amd", os.path.join(root, "__init__.py"), submodule_search_locations=[root])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["nimllm_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["nimllm_amd"]


# ---------------------------------------------------------------- the cases


def listed():
    return [
        # a CPU model's chat loop: host logits in, host id out, one at a time
        {"name": "chat_host_32k", "family": "chat", "rows": 1, "vocab": 32000},
        # one token of one context with the output matrix on the device
        {"name": "decode_q6k_1", "family": "decode", "rows": 1, "vocab": 128256, "cols": 2048, "type": "Q6_K"},
        # a small serving batch; an odd vocabulary, so rows start off 16 bytes
        {"name": "generate_24x50001", "family": "generate", "rows": 24, "vocab": 50001},
        # a large serving batch: the benchmark's headline workload
        {"name": "penalties_256x128k", "family": "penalties", "rows": 256, "vocab": 128256, "k": 50, "hist": 1024,
         "bias": 50},
        # no top-k: the reference's full sort with top-p and min-p
        {"name": "zipf_64x128k", "family": "zipf", "rows": 64, "vocab": 128256, "hist": 256},
        # a wide top-k over a flat row (creative settings)
        {"name": "topk1000_1024x128k", "family": "topk", "rows": 1024, "vocab": 128256, "k": 1000},
        # the largest batch: requests of all kinds together, heavy ties
        {"name": "mixed_2048x152k", "family": "mixed", "rows": 2048, "vocab": 151936, "hist": 512},
        # alternatives shown beside each token of a batch
        {"name": "toptokens_32x128k", "family": "toptokens", "rows": 32, "vocab": 128256, "n": 5},
        # whole distributions, for a program's own sampler
        {"name": "softmax_256x128k", "family": "softmax", "rows": 256, "vocab": 128256},
        # scoring a continuation, ragged in both sizes
        {"name": "logprob_201x50001", "family": "logprob", "rows": 201, "vocab": 50001},
        # perplexity of a chunk: the logits of every position, then their terms
        {"name": "perplexity_255x128k", "family": "perplexity", "rows": 255, "vocab": 128256, "cols": 2048,
         "type": "Q4_K"},
        # the output projection of an unquantised model, one token
        {"name": "head_f16_1", "family": "head", "rows": 1, "vocab": 128256, "cols": 2048, "type": "F16"},
    ]


_MOST_LOGITS = 2048 * 151936   # of the largest listed batch
_MOST_WEIGHTS = 128256 * 2048  # of the largest listed output matrix


def _spread(rng, lo, hi):
    """A whole number, even in its logarithm over lo .. hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["chat", "decode", "generate", "penalties", "zipf", "topk", "mixed", "toptokens", "softmax",
                         "logprob", "perplexity", "head"])
    vocab = _spread(rng, 8000, 151936)
    if rng.random() < 0.5:  # real vocabularies are often padded to a multiple of 64
        vocab = vocab // 64 * 64
    c = {"family": family, "vocab": vocab}
    if family == "chat":
        c["rows"] = 1
    elif family in ("decode", "perplexity", "head"):
        c["cols"] = rng.choice([1024, 2048, 3072, 4096])
        c["vocab"] = min(vocab, _MOST_WEIGHTS // c["cols"])
        if family == "perplexity":
            c["type"] = rng.choice(["Q4_K", "Q6_K"])
            c["rows"] = _spread(rng, 5, 255)
        elif family == "decode":
            c["type"] = rng.choice(["Q4_K", "Q6_K", "Q8_0"])
            c["rows"] = 1 if c["type"] == "Q8_0" else _spread(rng, 1, 24)
        else:
            c["type"] = rng.choice(["Q4_K", "Q6_K", "Q8_0", "F16"])
            c["rows"] = _spread(rng, 1, 4)
    elif family == "generate":
        c["rows"] = _spread(rng, 1, 256)
    elif family == "penalties":
        c.update(rows=_spread(rng, 1, 512), k=rng.choice([20, 40, 50, 64]), hist=_spread(rng, 16, 1024),
                 bias=rng.randrange(0, 51))
    elif family == "zipf":
        c.update(rows=_spread(rng, 1, 256), hist=_spread(rng, 16, 512))
    elif family == "topk":
        c.update(rows=_spread(rng, 1, 1024), k=rng.choice([10, 40, 64, 100, 300, 1000]))
    elif family == "mixed":
        c.update(rows=_spread(rng, 8, 2048), hist=_spread(rng, 16, 512))
    elif family == "toptokens":
        c.update(rows=_spread(rng, 1, 256), n=rng.choice([1, 5, 10, 20]))
    else:
        c["rows"] = _spread(rng, 1, 256)
    c["rows"] = max(1, min(c["rows"], _MOST_LOGITS // c["vocab"]))
    return c


# --------------------------------------------------------------- the inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(case, seed, scale):
    x = torch.randn(case["rows"], case["vocab"], generator=_gen(seed), device="cuda", dtype=torch.float32)
    return x.mul_(scale)


def _weights(case, seed):
    """GGUF rows of random blocks, scaled so that logits of unit hidden states
    spread as a model's do (a standard deviation of about 2 to 3), as flat bytes."""
    rows, cols, t, g = case["vocab"], case["cols"], case["type"], _gen(seed)
    if t == "F16":
        w = torch.empty(rows, cols, dtype=torch.float16, device="cuda")
        return w.normal_(0.0, 0.05, generator=g).view(torch.uint8).reshape(-1)
    block, size = {"Q4_K": (256, 144), "Q6_K": (256, 210), "Q8_0": (32, 34)}[t]
    n = rows * (cols // block)
    w = torch.randint(0, 256, (n, size), dtype=torch.uint8, generator=g, device="cuda")
    d = torch.rand(n, 1, generator=g, device="cuda") * 0.5 + 0.5
    if t == "Q6_K":
        w[:, 208:210] = (d * 1e-4).half().view(torch.uint8)
    elif t == "Q4_K":
        w[:, 0:2] = (d * 2.5e-4).half().view(torch.uint8)
        w[:, 2:4] = (d * 2.5e-4 * 7.5).half().view(torch.uint8)
    else:
        w[:, 0:2] = (d * 7e-4).half().view(torch.uint8)
    w = w.reshape(rows, -1)
    w[_end_ids(case)] = 0  # end-of-generation ids: logit 0, far below what is drawn (a run in mid-answer)
    return w.reshape(-1)


def _end_ids(case):
    return [2, case["vocab"] - 7]


def _zipf_history(rng, rows, n, vocab):
    """Ids that repeat as a text's do, each row over an order of its own."""
    z = rng.zipf(1.2, size=(rows, n)).astype(np.uint64) % np.uint64(1 << 40)
    step = rng.integers(1, 1 << 20, size=(rows, 1)).astype(np.uint64) * np.uint64(2) + np.uint64(1)
    return ((z * step) % np.uint64(vocab)).astype(np.int64)


def _default(m, seed):
    p = m.defaultSampling()
    p.seed = seed
    return p


def _contexts(m, case, seed):
    """generate_step's state for `rows` contexts in mid-answer, each with its own seed and last 64 ids."""
    B, V = case["rows"], case["vocab"]
    s = m.BatchSampler([_default(m, seed + b) for b in range(B)], V)
    s.accept(np.random.default_rng(seed).integers(0, V, size=(B, 64), dtype=np.int64))
    return {"sampler": s, "end": torch.tensor(_end_ids(case), dtype=torch.int32, device="cuda"),
            "done": torch.zeros(B, dtype=torch.int32, device="cuda")}


def _projection(m, case, seed):
    """The output matrix, the hidden states and the buffers a program keeps for nls_lm_head."""
    t = m.GGML_TYPES[case["type"]]
    need = m.lm_head_workspace(t, case["cols"], case["rows"])
    return {"weights": _weights(case, seed), "type": t,
            "hidden": torch.randn(case["rows"], case["cols"], generator=_gen(seed + 1), device="cuda"),
            "logits": torch.empty(case["rows"], case["vocab"], device="cuda"),
            "work": torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")}


def prepare(case, seed):
    m = _package()
    f, B, V = case["family"], case["rows"], case["vocab"]
    rng = np.random.default_rng(seed)
    s = {"m": m, "case": case, "run": _RUN[f]}
    if f == "chat":
        s["sampler"] = m.newSampler(_default(m, seed), V)
        for t in rng.integers(0, V, size=64):
            s["sampler"].accept(int(t))
        s["logits"] = (rng.standard_normal(V, dtype=np.float32) * np.float32(3.0))
    elif f == "decode":
        s.update(_projection(m, case, seed), **_contexts(m, case, seed))
    elif f in ("perplexity", "head"):
        s.update(_projection(m, case, seed))
        s["targets"] = torch.from_numpy(rng.integers(0, V, size=B, dtype=np.int32)).cuda()
    elif f == "generate":
        s.update(_contexts(m, case, seed), logits=_normal(case, seed, 3.0))
        s["logits"][:, _end_ids(case)] = -30.0
    elif f in ("penalties", "zipf", "topk", "mixed"):
        s["logits"], rows, hist = _RECIPES[f](m, case, seed, rng)
        s["sampler"] = m.BatchSampler(rows, V)
        if hist is not None:
            s["sampler"].accept(hist)
    else:
        s["logits"] = _normal(case, seed, 2.5)
        if f == "logprob":
            s["targets"] = torch.from_numpy(rng.integers(0, V, size=B, dtype=np.int32)).cuda()
    return s


def _penalties(m, case, seed, rng):
    B, V = case["rows"], case["vocab"]
    rows = []
    for b in range(B):
        ids = rng.choice(V, size=case["bias"], replace=False, shuffle=False)
        vals = rng.uniform(-5.0, 5.0, size=case["bias"])
        vals[:5] = -math.inf
        rows.append(m.SamplerParams(temperature=1.0, topK=case["k"], topP=0.95, repeatPenalty=1.0,
                                    presencePenalty=0.3, frequencyPenalty=0.5, seed=seed + b,
                                    logitBias=dict(zip(ids.tolist(), vals.tolist()))))
    return _normal(case, seed, 2.5), rows, _zipf_history(rng, B, case["hist"], V)


def _zipf(m, case, seed, rng):
    B, V = case["rows"], case["vocab"]
    x = _normal(case, seed, 1.0)
    g = _gen(seed + 1)
    for b in range(B):  # the rank of every id, at random
        x[b] -= 4.4 * torch.log(1.0 + torch.randperm(V, generator=g, device="cuda"))
    rows = [m.SamplerParams(temperature=0.7, topP=0.9, minP=0.05, repeatPenalty=1.1, seed=seed + b) for b in range(B)]
    return x, rows, rng.integers(0, V, size=(B, case["hist"]), dtype=np.int64)


def _topk(m, case, seed, rng):
    rows = [m.SamplerParams(temperature=1.2, topK=case["k"], topP=0.99, repeatPenalty=1.0, seed=seed + b)
            for b in range(case["rows"])]
    return _normal(case, seed, 1.0), rows, None


def _mixed(m, case, seed, rng):
    B, V = case["rows"], case["vocab"]
    kinds = [dict(temperature=0.0, topP=1.0), dict(temperature=1.0, topP=1.0, minP=0.1),
             dict(temperature=1.0, topP=1.0, topK=20), dict(temperature=1.0, topP=0.8)]
    rows = [m.SamplerParams(repeatPenalty=1.05, seed=seed + b, **kinds[k])
            for b, k in enumerate(rng.integers(0, 4, size=B))]
    x = _normal(case, seed, 8.0).round_().div_(4.0)
    return x, rows, rng.integers(0, V, size=(B, case["hist"]), dtype=np.int64)


_RECIPES = {"penalties": _penalties, "zipf": _zipf, "topk": _topk, "mixed": _mixed}


# ------------------------------------------------------------------ one pass


def _run_chat(s):
    t = s["sampler"].sample(s["logits"])
    s["sampler"].accept(t)
    return t


def _run_head(s):
    c = s["case"]
    return s["m"].lm_head(s["weights"], s["type"], c["vocab"], c["cols"], s["hidden"], out=s["logits"], work=s["work"])


def _run_decode(s):
    logits = _run_head(s)
    return {"logits": logits, "ids": s["sampler"].generate_step(logits, s["end"], s["done"])}


def _run_perplexity(s):
    logits = _run_head(s)
    return {"logits": logits, "nll": s["m"].row_nll_device(logits, s["targets"])}


def _run_generate(s):
    return s["sampler"].generate_step(s["logits"], s["end"], s["done"])


def _run_sample(s):
    return s["sampler"].sample(s["logits"])


def _run_toptokens(s):
    return s["m"].top_tokens_device(s["logits"], s["case"]["n"])


def _run_softmax(s):
    return s["m"].softmax_device(s["logits"])


def _run_logprob(s):
    return s["m"].log_prob_device(s["logits"], s["targets"])


_RUN = {"chat": _run_chat, "decode": _run_decode, "generate": _run_generate, "penalties": _run_sample,
        "zipf": _run_sample, "topk": _run_sample, "mixed": _run_sample, "toptokens": _run_toptokens,
        "softmax": _run_softmax, "logprob": _run_logprob, "perplexity": _run_perplexity, "head": _run_head}


def run(state):
    return state["run"](state)


# ------------------------------------------------------- bytes, bounds, oracle


def _matrix_bytes(case):
    return case["vocab"] * case["cols"] * {"Q4_K": 144 / 256, "Q6_K": 210 / 256, "Q8_0": 34 / 32, "F16": 2}[case["type"]]


def work(case):
    """Logits, weights, hidden states, the penalty window's ids (4 bytes), biases
    (8), uniforms (8) and ids (4) once each; the projection's products."""
    f, B, V = case["family"], case["rows"], case["vocab"]
    rows = 4 * B * V
    if f in ("decode", "perplexity", "head"):
        b = _matrix_bytes(case) + 4 * B * case["cols"] + rows  # the logits are an output: written
        b += {"decode": B * (4 * 64 + 12), "perplexity": 12 * B, "head": 0}[f]
        return {"bytes": b, "flops": 2.0 * B * V * case["cols"]}
    window = 64 if f in ("chat", "generate") else case.get("hist", 0)
    extra = {"toptokens": 8 * case.get("n", 0), "softmax": 4 * V, "logprob": 16}
    return {"bytes": rows + B * extra.get(f, 12 + 4 * window + 8 * case.get("bias", 0)), "flops": 0.0}


def tolerance(case):
    """Ids and every fp32 result are the reference's own, bit for bit (its fp32
    operations in its order).  logprob's logarithm and perplexity's terms are
    float64 sums and logarithms in no fixed order, which come within 1e-13."""
    return {"rel": 1e-12} if case["family"] in ("logprob", "perplexity") else "exact"


def _dequantised(case, w):
    """The weights [vocab, cols] in float64."""
    rows, cols, t = case["vocab"], case["cols"], case["type"]
    if t == "F16":
        return w.view(torch.float16).reshape(rows, cols).double()

    def half(b):
        return b.contiguous().view(torch.float16).double()

    if t == "Q8_0":
        b = w.reshape(-1, 34)
        return (half(b[:, 0:2]) * b[:, 2:].view(torch.int8).double()).reshape(rows, cols)
    if t == "Q4_K":  # d, dmin, eight 6-bit (scale, min) pairs, nibbles by pairs of 32
        b = w.reshape(-1, 144)
        s = b[:, 4:16].int()
        lo, hi = s[:, 0:4], s[:, 4:8]
        scale = torch.cat([lo & 63, (s[:, 8:12] & 15) | ((lo >> 6) << 4)], 1)
        least = torch.cat([hi & 63, (s[:, 8:12] >> 4) | ((hi >> 6) << 4)], 1)
        q = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        return ((half(b[:, 0:2]) * scale).unsqueeze(2) * q - (half(b[:, 2:4]) * least).unsqueeze(2)).reshape(rows, cols)
    b = w.reshape(-1, 210)  # Q6_K: low nibbles, high bit pairs, sixteen int8 scales, d
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    low = torch.cat([ql & 15, ql >> 4], 2)                                          # [n, half, quarter, 32]
    high = torch.stack([(qh >> k) & 3 for k in (0, 2, 4, 6)], 2)
    q = (low | (high << 4)).double().reshape(-1, 16, 16) - 32.0
    scale = b[:, 192:208].contiguous().view(torch.int8).double() * half(b[:, 208:210])
    return (scale.unsqueeze(2) * q).reshape(rows, cols)


def _logits64(case, s):
    """The projection in 64 bits: of the hidden states rounded to 8 bits by
    blocks where that is what is computed, else of the hidden states."""
    x = s["hidden"].double()
    block = {"Q4_K": 256, "Q6_K": 256, "Q8_0": 32, "F16": 0}[case["type"]]
    if block:
        x = x.reshape(case["rows"], -1, block)
        d = x.abs().amax(2, keepdim=True) / 127.0
        x = (torch.sign(x) * torch.floor((x / d).abs() + 0.5) * d).reshape(case["rows"], -1)
    out = torch.empty(case["rows"], case["vocab"], dtype=torch.float64, device="cuda")
    w, per = s["weights"].reshape(case["vocab"], -1), 16384
    for r in range(0, case["vocab"], per):  # 16384 rows at a time: 0.5 GB of float64 weights at most
        part = w[r:r + per].contiguous()
        out[:, r:r + per] = x @ _dequantised(dict(case, vocab=part.shape[0]), part.reshape(-1)).t().contiguous()
    return out


def _nll64(logits, targets):
    return torch.logsumexp(logits, 1) - logits.gather(1, targets.long().reshape(-1, 1)).reshape(-1)


def exact(case, seed):
    f = case["family"]
    if f in ("chat", "generate", "penalties", "zipf", "topk", "mixed"):
        return None  # ids only
    s = prepare(case, seed)
    if f in ("decode", "perplexity", "head"):
        y = _logits64(case, s)
        if f == "perplexity":
            return {"logits": y, "nll": _nll64(y, s["targets"])}
        return {"logits": y, "ids": None} if f == "decode" else y
    x = s["logits"].double()
    if f == "toptokens":
        return (None, torch.softmax(x, 1).topk(min(case["n"], case["vocab"]), 1).values)
    if f == "softmax":
        return torch.softmax(x, 1)
    logp = -_nll64(x, s["targets"])
    return (torch.exp(logp), logp)
