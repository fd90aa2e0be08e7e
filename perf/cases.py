"""The work that the framework is measured on.

Six kinds of call, each through the package's public entry points, over the
sizes in which programs make them:

* ``loop``   -- the AR loop's sampling: one ``sample_rows`` call a step with the
  history kept on the device as a set, a number of steps captured into one
  graph as a decode loop captures them, each step with logits of its own.
* ``rows``   -- one ``sample_rows`` call at a vocabulary of the semantic head's
  size, histories as lists of ids.
* ``big``    -- one ``sample_rows`` call at a text model's vocabulary.
* ``head``   -- the final LayerNorm and LM head alone (logits out).
* ``step``   -- ``lmhead_sample``: the hidden rows to logits and tokens.
* ``stream`` -- ``sample_stream``: many AR steps of known logits in one call.

Sampling parameters (``preset``): ``defaults`` the TTS pipeline's own on every
row, ``assorted`` every row its own, ``nucleus`` top_p alone, ``topk`` top_k 50
and top_p 0.95, ``ties`` top_p 0.5 on rows a tenth of whose values are equal to
the maximum (logits of few significant bits), ``greedy`` argmax.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("mlx-confucius4-tts_amd"))
import c4s  # noqa: E402

SEMANTIC_VOCAB = 8194
STOP_TOKEN = 8193
DEFAULT_SEED = 1234


def listed():
    return [
        # One utterance: the product's usual call, where latency is everything.
        {"name": "loop_1_defaults", "kind": "loop", "rows": 1, "vocab": 8194, "steps": 32, "preset": "defaults",
         "dtype": "f32"},
        # A batch of requests, each with its own sampling parameters.
        {"name": "loop_64_assorted", "kind": "loop", "rows": 64, "vocab": 8194, "steps": 32, "preset": "assorted",
         "dtype": "f32"},
        # A large offline batch, every row its own parameters.
        {"name": "rows_1000_assorted", "kind": "rows", "rows": 1000, "vocab": 8194, "preset": "assorted",
         "dtype": "f32"},
        # bf16 logits, many of them equal: the nucleus cut falls among ties.
        {"name": "rows_1024_ties_bf16", "kind": "rows", "rows": 1024, "vocab": 8194, "preset": "ties", "dtype": "bf16"},
        # A text model's vocabulary, the usual top_k + top_p.
        {"name": "big_256_topk", "kind": "big", "rows": 256, "vocab": 151936, "preset": "topk", "dtype": "f32"},
        # The same vocabulary without top_k, on the bf16 logits that such a model's head gives.
        {"name": "big_32_nucleus_bf16", "kind": "big", "rows": 32, "vocab": 151936, "preset": "nucleus",
         "dtype": "bf16"},
        # The head of a single utterance in the reference's own weight type.
        {"name": "head_1_f32", "kind": "head", "rows": 1, "dim": 1280, "vocab": 8194, "weight": "f32"},
        # The head of a batch, bf16 weights.
        {"name": "head_64_bf16", "kind": "head", "rows": 64, "dim": 1280, "vocab": 8194, "weight": "bf16"},
        # The head of a batch, 8-bit weights in groups of 64.
        {"name": "head_64_q8", "kind": "head", "rows": 64, "dim": 1280, "vocab": 8194, "weight": "q8"},
        # Logits of many positions at once (scoring given sequences), an odd number of them.
        {"name": "head_777_bf16", "kind": "head", "rows": 777, "dim": 1280, "vocab": 8194, "weight": "bf16"},
        # One whole AR step behind the model's last layer, in the reference's own weight type.
        {"name": "step_64_f32", "kind": "step", "rows": 64, "dim": 1280, "vocab": 8194, "weight": "f32",
         "preset": "assorted"},
        # A thousand steps of a batch with known logits (replaying recorded ones).
        {"name": "stream_64x1000", "kind": "stream", "rows": 64, "vocab": 8194, "steps": 1000, "preset": "assorted"},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["loop", "rows", "rows", "big", "big", "head", "head", "step", "stream"])
    # half of the draws at the semantic vocabulary, the others anywhere in the range
    v = SEMANTIC_VOCAB if rng.random() < 0.5 else _log(rng, 500, 12288)
    if kind == "loop":
        return {"kind": kind, "rows": _log(rng, 1, 128), "vocab": v, "steps": rng.randint(8, 32),
                "preset": rng.choice(["defaults", "assorted", "nucleus", "greedy"]),
                "dtype": rng.choice(["f32", "f32", "bf16"])}
    if kind == "rows":
        return {"kind": kind, "rows": _log(rng, 1, 1024), "vocab": v,
                "preset": rng.choice(["defaults", "assorted", "nucleus", "ties", "greedy"]),
                "dtype": rng.choice(["f32", "bf16"])}
    if kind == "big":
        v = _log(rng, 12289, 262144)
        return {"kind": kind, "rows": min(_log(rng, 1, 256), 256 * 151936 // v), "vocab": v,
                "preset": rng.choice(["topk", "nucleus", "greedy"]), "dtype": rng.choice(["f32", "bf16"])}
    if kind == "stream":
        rows = _log(rng, 1, 64)
        return {"kind": kind, "rows": rows, "vocab": min(v, SEMANTIC_VOCAB), "steps": _log(rng, 64, 1000),
                "preset": rng.choice(["defaults", "assorted"])}
    dim = 128 * rng.randint(2, 16)
    weight = rng.choice(["bf16", "f32", "q8"])
    if kind == "step":
        return {"kind": kind, "rows": _log(rng, 1, 200), "dim": dim, "vocab": v, "weight": weight,
                "preset": rng.choice(["defaults", "assorted", "nucleus"])}
    return {"kind": kind, "rows": _log(rng, 1, 1000), "dim": dim, "vocab": v, "weight": weight}


# ---- inputs ----------------------------------------------------------------------

_context = _queue = None


def _ctx():
    """The program's library context (one per host thread) and the stream that it gives the long calls."""
    global _context, _queue
    if _context is None:
        _context, _queue = c4s.Context(0), torch.cuda.Stream()
    return _context, _queue


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _semantic_logits(g, lead, vocab, preset, dtype):
    """[*lead, vocab]: N(0, 3^2) with five ids at +12 (a peaked step); `ties`: heavy-tailed
    values of bf16 precision, a tenth of each row's ids at the row's maximum."""
    x = torch.randn((*lead, vocab), generator=g, device="cuda")
    if preset == "ties":
        den = torch.randn((3, *lead, vocab), generator=g, device="cuda").square_().mean(dim=0).sqrt_()
        x = (x.mul_(4.0) / den).to(torch.bfloat16)   # Student-t, three degrees of freedom
        at = torch.rand((*lead, vocab), generator=g, device="cuda") < 0.1
        x = torch.where(at, x.amax(dim=-1, keepdim=True), x)
        return x if dtype == "bf16" else x.float()
    x.mul_(3.0)
    x.scatter_(-1, torch.randint(0, vocab, (*lead, 5), generator=g, device="cuda"), 12.0)
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _text_logits(g, rows, vocab, dtype):
    """[rows, vocab]: N(0, 2^2) plus 10 (rank + 1)^-1.1 over a random order of the ids."""
    x = torch.randn((rows, vocab), generator=g, device="cuda").mul_(2.0)
    boost = 10.0 * torch.arange(1, vocab + 1, device="cuda", dtype=torch.float64).pow_(-1.1)
    boost = boost.float()
    for r in range(rows):
        x[r] += boost[torch.randperm(vocab, generator=g, device="cuda")]
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _params(seed, rows, vocab, preset, h_lo=50, h_hi=800):
    """History lists, per-row sampling parameters and generator states."""
    c = torch.Generator()
    c.manual_seed(seed)

    def pick(values, dtype):
        return torch.tensor(values, dtype=dtype)[torch.randint(0, len(values), (rows,), generator=c)]

    if preset == "assorted":
        temp = 0.6 + 0.6 * torch.rand(rows, generator=c)
        top_k, top_p = pick([0, 20, 30, 50], torch.int32), pick([1.0, 0.9, 0.8], torch.float32)
        pen = pick([1.0, 10.0], torch.float32)
    else:
        t, k, p, w = {"defaults": (0.8, 30, 0.8, 10.0), "nucleus": (0.8, 0, 0.9, 1.2), "topk": (0.7, 50, 0.95, 1.2),
                      "ties": (1.0, 0, 0.5, 10.0), "greedy": (1.0, 0, 1.0, 1.2)}[preset]
        temp, top_p, pen = (torch.full((rows,), v, dtype=torch.float32) for v in (t, p, w))
        top_k = torch.full((rows,), k, dtype=torch.int32)
    lens = torch.randint(h_lo, h_hi + 1, (rows,), generator=c)
    off = torch.zeros(rows + 1, dtype=torch.int64)
    off[1:] = lens.cumsum(0)
    ids = torch.randint(0, vocab, (int(off[-1]),), generator=c, dtype=torch.int32)
    do = torch.full((rows,), 0 if preset == "greedy" else 1, dtype=torch.uint8)
    base = int(torch.randint(1, 1 << 62, (1,), generator=c))
    rng = torch.tensor([(base + b * 0x100000001B3) & ((1 << 63) - 1) for b in range(rows)], dtype=torch.int64)
    return {"ids": ids.cuda(), "off": off.cuda(), "temp": temp.cuda(), "top_k": top_k.cuda(), "top_p": top_p.cuda(),
            "pen": pen.cuda(), "do": do.cuda(), "rng": rng.cuda()}


def _head(case, seed):
    """Hidden rows, LayerNorm and head tensors; 8-bit weights as codes with a scale and offset a group of 64."""
    g = _gen(seed)
    rows, dim, vocab = case["rows"], case["dim"], case["vocab"]
    w = torch.randn((vocab, dim), generator=g, device="cuda").mul_(0.02)
    h = {"hidden": torch.randn((rows, dim), generator=g, device="cuda").to(torch.bfloat16),
         "gamma": torch.randn(dim, generator=g, device="cuda").mul_(0.02).add_(1.0),
         "beta": torch.randn(dim, generator=g, device="cuda").mul_(0.02),
         "bias": torch.randn(vocab, generator=g, device="cuda").mul_(0.02), "quant": None}
    if case["weight"] == "q8":
        grp = w.view(vocab, dim // 64, 64)
        lo, hi = grp.amin(dim=2), grp.amax(dim=2)
        scale = torch.where(hi > lo, (hi - lo) / 255.0, torch.ones_like(hi))
        q = torch.clamp(torch.round((grp - lo[..., None]) / scale[..., None]), 0, 255)
        h["weight"] = q.to(torch.uint8).view(vocab, dim)
        h["quant"] = (scale.contiguous(), lo.contiguous(), 64)
    else:
        h["weight"] = w.to(torch.bfloat16) if case["weight"] == "bf16" else w
    return h


def _stop(case):
    """The end token where the vocabulary has it."""
    return STOP_TOKEN if case["vocab"] > STOP_TOKEN else case["vocab"] - 1


def prepare(case, seed):
    kind, rows, vocab = case["kind"], case["rows"], case["vocab"]
    ctx, queue = _ctx()
    s = {"kind": kind, "ctx": ctx, "queue": queue, "stop": _stop(case)}
    if kind in ("head", "step"):
        s.update(_head(case, seed))
        s["logits"] = torch.empty((rows, vocab), device="cuda")
        if kind == "step":
            s.update(_params(seed, rows, vocab, case["preset"]))
            s["tokens"] = torch.empty(rows, dtype=torch.int32, device="cuda")
        return s
    g = _gen(seed)
    if kind == "big":
        s.update(_params(seed, rows, vocab, case["preset"], 2048, 2048))
        s["logits"] = _text_logits(g, rows, vocab, case["dtype"])
    else:
        s.update(_params(seed, rows, vocab, case["preset"], *((1000, 1000) if case["preset"] == "ties" else (50, 800))))
        lead = (rows,) if kind == "rows" else (case["steps"], rows)
        s["logits"] = _semantic_logits(g, lead, vocab, case["preset"], case.get("dtype", "f32"))
    s["tokens"] = torch.empty(s["logits"].shape[:-1], dtype=torch.int32, device="cuda")
    if kind == "loop":
        s["bits"] = torch.empty((rows, (vocab + 31) // 32), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=queue):
            _steps(s, case["steps"])
    return s


def _steps(s, n):
    """A new utterance's first n AR steps on the current stream: the history set, then a call a step."""
    rows, vocab = s["logits"].shape[1:]
    s["ctx"].hist_bits_init(s["ids"], s["off"], rows, vocab, s["bits"])
    for i in range(n):
        s["ctx"].sample_rows(s["logits"][i], None, None, s["temp"], s["top_k"], s["top_p"], s["pen"], s["rng"],
                             s["tokens"][i], do_sample=s["do"], hist_bits=s["bits"], stop_token=s["stop"])


# ---- one pass ---------------------------------------------------------------------

def run(s):
    kind, ctx = s["kind"], s["ctx"]
    if kind == "loop":
        s["graph"].replay()
        return {"tokens": s["tokens"], "rng": s["rng"], "history": s["bits"]}
    if kind == "head":
        ctx.lmhead(s["hidden"], s["gamma"], s["beta"], s["weight"], s["bias"], s["logits"], quant=s["quant"])
        return {"logits": s["logits"]}
    if kind == "step":
        ctx.lmhead_sample(s["hidden"], s["gamma"], s["beta"], s["weight"], s["bias"], s["ids"], s["off"], s["temp"],
                          s["top_k"], s["top_p"], s["pen"], s["rng"], s["tokens"], logits=s["logits"],
                          do_sample=s["do"], quant=s["quant"])
        return {"logits": s["logits"], "tokens": s["tokens"], "rng": s["rng"]}
    if kind == "stream":
        ctx.sample_stream(s["logits"], s["ids"], s["off"], s["temp"], s["top_k"], s["top_p"], s["pen"], s["rng"],
                          s["tokens"], do_sample=s["do"], stop_token=-1, stream=s["queue"])
        return {"tokens": s["tokens"], "rng": s["rng"]}
    ctx.sample_rows(s["logits"], s["ids"], s["off"], s["temp"], s["top_k"], s["top_p"], s["pen"], s["rng"],
                    s["tokens"], do_sample=s["do"])
    return {"tokens": s["tokens"], "rng": s["rng"]}


# ---- what a pass cannot do without --------------------------------------------------

def work(case):
    kind, rows, vocab = case["kind"], case["rows"], case["vocab"]
    if kind in ("head", "step"):
        dim = case["dim"]
        per = {"bf16": 2.0, "f32": 4.0, "q8": 1.0 + 8.0 / 64}[case["weight"]]
        nbytes = per * vocab * dim + 2 * rows * dim + 4 * vocab + 8 * dim + 4 * rows * vocab
        if kind == "step":
            nbytes += rows * (4 * 425 + 45)
        return {"bytes": nbytes, "flops": 2.0 * rows * dim * vocab}
    size = 2 if case.get("dtype") == "bf16" else 4
    # the parameters and the generator state in and out, the token out
    if kind == "loop":   # the set of ids read and its word updated each step
        words = 4 * ((vocab + 31) // 32)
        return {"bytes": float(case["steps"] * rows * (size * vocab + words + 8 + 37)), "flops": 0.0}
    hist = 4 * (2048 if kind == "big" else 1000 if case["preset"] == "ties" else 425)
    if kind == "stream":
        return {"bytes": float(case["steps"] * rows * (4 * vocab + 4) + rows * (hist + 41)), "flops": 0.0}
    return {"bytes": float(rows * (size * vocab + hist + 45)), "flops": 0.0}


# The head's rows are bf16 and its sums float32. Against 64 bits its 2-norm error is 2.4e-6 to 2.5e-6 of the
# logits for bf16 and float32 weights, and 7.5e-6 to 9e-6 for 8-bit weights (codes up to 255 that the group's
# offset cancels): four times that. Tokens, generator states and history sets are whole numbers and stay as they
# are; behind the head a logit's last bit may move a draw.
def tolerance(case):
    if case["kind"] not in ("head", "step"):
        return "exact"
    rel = 4e-5 if case["weight"] == "q8" else 1e-5
    return {"rel": rel} if case["kind"] == "head" else {"rel": rel, "differ": 0.01}


def exact(case, seed):
    """The head's logits in 64 bits; tokens and generator states have no such value."""
    if case["kind"] not in ("head", "step"):
        return None
    h = _head(case, seed)
    x = h["hidden"].double()
    x = x - x.mean(dim=1, keepdim=True)
    x = x / (x.square().mean(dim=1, keepdim=True) + 1e-5).sqrt()
    x = x * h["gamma"].double() + h["beta"].double()
    w = h["weight"].double()
    if h["quant"] is not None:
        scale, lo, group = h["quant"]
        rows, groups = scale.shape
        w = (w.view(rows, groups, group) * scale.double()[..., None] + lo.double()[..., None]).view(rows, -1)
    logits = x @ w.t() + h["bias"].double()
    return {"logits": logits} if case["kind"] == "head" else {"logits": logits, "tokens": None, "rng": None}
