"""The work that programs built on this backend hand it, as cases that can be timed.

A case is one call, or one request made of a few calls, through the public
entry points (``HipBackend``, ``HipModel``, ``HipBatch``):

``linear``    one linear layer through the operator interface: y = x . W^T
``step``      one decode step with its logits (a token loop that samples on the host)
``prompt``    the prompt rows of one request in one forward, with the last row's logits
``generate``  a request: its prompt, then a number of tokens from the resident loop
``batch``     several requests decoded together

The widths are those of the measured workloads (the 1B, 8B and 70B Llama
shapes), the decoder cut to a few of its layers so that a case holds what each
layer and the head do; the small width is the one of the parity tests.
Weights are uniform 4-bit or 8-bit codes with the scales of the synthetic
workloads, activations and caches normal.  Where a case returns tokens of the
greedy loop, the codes are centred and the head is drawn from the embedding, so
that the top token stands clear of the others, as a trained model's does:
otherwise a last-bit difference in one step would decide which text is compared.
"""
from __future__ import annotations

import importlib
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "llm.rs_amd"))
lh = importlib.import_module("llmrs_hip")

DEV = "cuda" if torch.cuda.is_available() else "cpu"

# name: (query heads, KV heads, head_dim, ffn); hidden = query heads * head_dim
WIDTHS = {
    "small": (4, 2, 64, 512),
    "1b": (32, 8, 64, 8192),
    "8b": (32, 8, 128, 14336),
    "70b": (64, 8, 128, 28672),
}
SCALES = {"q4": (0.003, 0.006), "q4_0": (0.003, 0.006), "q8_0": (2e-4, 3.5e-4)}
DTYPES = {"q4": lh.DType.Q4, "q4_0": lh.DType.Q4_0, "q8_0": lh.DType.Q8_0}
SLOTS = (lh.W_Q, lh.W_K, lh.W_V, lh.W_O, lh.W_GATE, lh.W_UP, lh.W_DOWN)
THETA, EPS = 500000.0, 1e-5


def _model(kind, name, width, layers, vocab, weight, kv, rows, start=0, steps=0, batch=0, order="fast", sampled=False):
    return {"name": name, "kind": kind, "width": width, "layers": layers, "vocab": vocab, "weight": weight, "kv": kv,
            "rows": rows, "start": start, "steps": steps, "batch": batch, "order": order, "sampled": sampled}


def listed():
    return [
        # the smallest call: one row through one small linear layer, as a host-driven layer loop makes it
        {"name": "linear_row", "kind": "linear", "rows": 1, "n": 2048, "k": 2048, "weight": "q4_0"},
        # the same call for the rows of a short prompt, at the 8B width
        {"name": "linear_rows", "kind": "linear", "rows": 48, "n": 4096, "k": 4096, "weight": "q4_0"},
        # a chat request on the small shape with the exact cache: 32 prompt tokens, 64 tokens of greedy reply
        _model("generate", "generate_1b_f32kv", "1b", 4, 32000, "q4_0", "f32", 32, steps=64),
        # the host-side sampler's token loop at the 8B width, full vocabulary, an ordinary context
        _model("step", "step_8b", "8b", 2, 128256, "q4_0", "f16", 1, start=700),
        # the same loop where the logits must be the reference's bit for bit
        _model("step", "step_8b_reforder", "8b", 2, 32000, "q4_0", "f16", 1, start=550, order="reference"),
        # decoding deep in a long document, the largest width
        _model("step", "step_70b_8192", "70b", 1, 32000, "q4_0", "f16", 1, start=8192),
        # a short question to a model loaded from safetensors (f32 scales)
        _model("prompt", "prompt_8b_23", "8b", 2, 32000, "q4", "f16", 23),
        # the second turn of a chat: 77 rows after 300 cached positions, 8-bit weights
        _model("prompt", "prompt_1b_q8_77", "1b", 2, 32000, "q8_0", "f16", 77, start=300),
        # a page of text on the small shape with the exact cache
        _model("prompt", "prompt_1b_f32kv_700", "1b", 4, 32000, "q4_0", "f32", 700),
        # the largest: a whole prefill chunk at the 8B width
        _model("prompt", "prompt_8b_2048", "8b", 2, 32000, "q4_0", "f16", 2048),
        # a sampled reply in the reference's operation order: repeatable text
        _model("generate", "generate_8b_sampled", "8b", 2, 32000, "q4_0", "f16", 130, steps=16, order="reference",
               sampled=True),
        # sixteen requests with prompts of different lengths served together
        _model("batch", "batch_8b_16", "8b", 2, 32000, "q4_0", "f16", 40, steps=24, batch=16),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["linear", "step", "step", "prompt", "prompt", "prompt", "generate", "batch"])
    if kind == "linear":
        return {"kind": "linear", "rows": log_int(1, 256), "n": 32 * log_int(16, 448), "k": 32 * log_int(16, 448),
                "weight": rng.choice(["q4", "q4_0", "q8_0"])}
    width = rng.choice(["small", "1b", "1b", "8b", "8b", "8b", "70b"])
    weight = rng.choice(["q4", "q4_0", "q4_0", "q8_0"])
    kv = rng.choice(["f16", "f16", "f32"])
    layers = 1 if width in ("70b", "8b") else rng.randint(1, 2)
    vocab = rng.choice([1000, 32000, 32000]) if width == "small" else 32000
    order = rng.choice(["fast", "fast", "reference"])
    if kind == "step":
        return _pick(_model(kind, "", width, layers, vocab, weight, kv, 1, start=log_int(1, 8192), order=order))
    if kind == "prompt":
        # the small widths take whole chunks in either order; the largest width, and the reference order's
        # attention (one score at a time), are met with shorter prompts
        most = 512 if width == "70b" or order == "reference" else 2048
        return _pick(_model(kind, "", width, layers, vocab, weight, kv, log_int(2, most),
                            start=rng.choice([0, 0, log_int(1, 1024)]), order=order))
    if kind == "generate":
        sampled = rng.random() < 0.5
        return _pick(_model(kind, "", width, layers, vocab, weight, kv, log_int(1, 256), steps=log_int(2, 48),
                            order="reference" if sampled else order, sampled=sampled))
    return _pick(_model(kind, "", width if width != "70b" else "8b", 1, vocab, weight, kv, log_int(4, 48),
                        steps=log_int(2, 24), batch=log_int(2, 40)))


def _pick(case):
    return {k: v for k, v in case.items() if k != "name"}


# ---- inputs ----------------------------------------------------------------
def _gen(seed, *tag):
    h = 1469598103934665603
    for t in (seed,) + tag:
        h = ((h ^ (int(t) & 0xFFFFFFFF)) * 1099511628211) & 0x7FFFFFFFFFFFFFFF
    g = torch.Generator(device=DEV)
    g.manual_seed(h)
    return g


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std + mean


def _host(t):
    return t.cpu().numpy()


def _scales(g, weight, n, k):
    lo, hi = SCALES[weight]
    s = torch.rand(n, k // 32, generator=g, device=DEV) * (hi - lo) + lo
    return s if weight == "q4" else s.half().float()


def _codes(g, weight, n, k, centred=False):
    """Uniform codes: [n][k/2] packed nibbles (element 2i the low one of byte i; centred: 1 to 15, so that
    their mean is the format's zero, 8), or [n][k] int8."""
    if weight == "q8_0":
        return torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    if centred:
        q = torch.randint(1, 16, (n, k), generator=g, device=DEV, dtype=torch.uint8)
        return q[:, 0::2] | (q[:, 1::2] << 4)
    return torch.randint(0, 256, (n, k // 2), generator=g, device=DEV, dtype=torch.uint8)


def _quantised(w, weight):
    """Codes and scales nearest to the f32 matrix w (blocks of 32)."""
    n, k = w.shape
    b = w.reshape(n, k // 32, 32)
    top = 127.0 if weight == "q8_0" else 7.0
    s = b.abs().amax(-1) / top
    s = s if weight == "q4" else s.half().float()
    q = torch.where(s[..., None] > 0, torch.round(b / s[..., None].clamp_min(1e-30)), torch.zeros_like(b)).clamp(-top, top)
    q = q.reshape(n, k)
    if weight == "q8_0":
        return q.to(torch.int8), s
    u = (q + 8).to(torch.uint8)
    return u[:, 0::2] | (u[:, 1::2] << 4), s


def _value(codes, scales, weight):
    """The matrix that codes and scales stand for, in 64 bits."""
    n = codes.shape[0]
    if weight == "q8_0":
        q = codes.double()
    else:
        q = torch.stack((codes & 15, codes >> 4), -1).reshape(n, -1).double() - 8
    k = q.shape[1]
    return (q.reshape(n, k // 32, 32) * scales.double()[..., None]).reshape(n, k)


def _shape(case, slot):
    nq, nkv, hd, ffn = WIDTHS[case["width"]]
    H = nq * hd
    return {lh.W_Q: (H, H), lh.W_K: (nkv * hd, H), lh.W_V: (nkv * hd, H), lh.W_O: (H, H), lh.W_GATE: (ffn, H),
            lh.W_UP: (ffn, H), lh.W_DOWN: (H, ffn), lh.W_LM_HEAD: (case["vocab"], H)}[slot]


def _linear(case, seed, layer, slot):
    n, k = _shape(case, slot)
    g = _gen(seed, 1, layer + 1, slot)
    return _codes(g, case["weight"], n, k, _peaked(case)), _scales(g, case["weight"], n, k)


def _peaked(case):
    """Whether the head is drawn from the embedding: the greedy loops."""
    return case["kind"] in ("generate", "batch") and not case["sampled"]


def _embedding(case, seed):
    H = _shape(case, lh.W_O)[0]
    return _normal(_gen(seed, 2), case["vocab"], H, std=2.0 if _peaked(case) else 0.02)


def _lm_head(case, seed, embed):
    if not _peaked(case):
        return _linear(case, seed, -1, lh.W_LM_HEAD)
    # row t + 1 holds the direction of token t, in noise of half its size
    w = torch.roll(embed, 1, 0) * 0.5 + _normal(_gen(seed, 3), *embed.shape, std=0.5)
    return _quantised(w * 0.02, case["weight"])


def _norm(case, seed, layer, slot):
    return _normal(_gen(seed, 4, layer + 1, slot), _shape(case, lh.W_O)[0], mean=1.0, std=0.02)


def _tokens(case, seed, slot=0):
    g = torch.Generator()
    g.manual_seed(int(seed) * 1000003 + 77 * slot + 5)
    rows = case["rows"]
    if case["kind"] == "batch":  # prompts of different lengths, up to `rows`
        rows = 1 + (7919 * (slot + 1)) % rows
    return torch.randint(0, case["vocab"], (rows,), generator=g, dtype=torch.int32)


def _cache(case, seed, layer):
    """K (as rotated) and V of the cached positions, [KV heads][start][head_dim]."""
    nq, nkv, hd, _ = WIDTHS[case["width"]]
    g = _gen(seed, 5, layer)
    return _normal(g, nkv, case["start"], hd), _normal(g, nkv, case["start"], hd)


def _settle():
    """Takes the "not found" that looking a kernel up in one code object after another leaves as this
    thread's last HIP error, which torch would report at its own next launch."""
    try:
        torch.zeros(1, device=DEV)
    except RuntimeError as e:
        if "not found" not in str(e):
            raise


def prepare(case, seed):
    _settle()
    if case["kind"] == "linear":
        be = lh.HipBackend()
        _settle()
        g = _gen(seed, 1)
        codes = _host(_codes(g, case["weight"], case["n"], case["k"]))
        scales = _host(_scales(g, case["weight"], case["n"], case["k"]))
        make = lh.Tensor.from_q8_0 if case["weight"] == "q8_0" else lh.Tensor.from_q4
        x = _host(_normal(_gen(seed, 6), case["rows"], case["k"]))
        return {"case": case, "be": be, "x": lh.Tensor.from_numpy(x), "w": make(codes, scales, case["n"], case["k"])}
    nq, nkv, hd, ffn = WIDTHS[case["width"]]
    kv = lh.DType.F32 if case["kv"] == "f32" else lh.DType.F16
    room = case["start"] + case["rows"] + case["steps"] + 1
    m = lh.HipModel(lh.ModelConfig(case["layers"], nq * hd, nq, nkv, hd, ffn, case["vocab"], room, EPS, THETA,
                                   int(DTYPES[case["weight"]]), int(kv)))
    _settle()
    put = m.set_linear_q8_0 if case["weight"] == "q8_0" else m.set_linear_q4
    embed = _embedding(case, seed)
    m.set_embedding(_host(embed))
    m.set_norm(-1, lh.N_FINAL, _host(_norm(case, seed, -1, 0)))
    put(-1, lh.W_LM_HEAD, *(_host(t) for t in _lm_head(case, seed, embed)))
    for layer in range(case["layers"]):
        for slot in (lh.N_INPUT, lh.N_POST):
            m.set_norm(layer, slot, _host(_norm(case, seed, layer, slot)))
        for slot in SLOTS:
            put(layer, slot, *(_host(t) for t in _linear(case, seed, layer, slot)))
        if case["start"]:
            k, v = (_host(t) for t in _cache(case, seed, layer))
            for head in range(nkv):
                m.kv_write(layer, head, 0, k[head], v[head])
    if case["order"] == "reference":
        m.set_exact(True)
    if case["sampled"]:
        m.set_sampling(lh.Sampling.make(seed=int(seed), eos=()))
    state = {"case": case, "model": m}
    if case["kind"] == "batch":
        state["prompts"] = [_tokens(case, seed, s).numpy() for s in range(case["batch"])]
        state["batch"] = lh.HipBatch(m, case["batch"])
    else:
        state["tokens"] = _tokens(case, seed).numpy()
    return state


# ---- one pass --------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        return state["be"].matmul_transposed(state["x"], state["w"]).data()
    m = state["model"]
    if case["kind"] in ("step", "prompt"):
        logits, _, _ = m.forward(state["tokens"], case["start"])
        return {"logits": logits}
    if case["kind"] == "generate":
        tokens = m.generate(state["tokens"], case["steps"])
        logits, _, _ = m.forward(tokens[-1:], state["tokens"].size + tokens.size - 1)
        return {"tokens": tokens, "logits": logits}
    b = state["batch"]
    for slot, prompt in enumerate(state["prompts"]):
        b.begin(slot, prompt)
    b.decode_steps(case["steps"])
    tokens = [b.tokens(slot, prompt.size + case["steps"] + 1) for slot, prompt in enumerate(state["prompts"])]
    return {"tokens": np.concatenate(tokens), "logits": b.logits()}


# ---- what a pass cannot do without ------------------------------------------
def _per_weight(case):
    return {"q4": 20 / 32, "q4_0": 18 / 32, "q8_0": 34 / 32}[case["weight"]]


def work(case):
    if case["kind"] == "linear":
        r, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k * _per_weight(case) + 4 * r * (n + k), "flops": 2 * r * n * k}
    nq, nkv, hd, ffn = WIDTHS[case["width"]]
    H, L, V = nq * hd, case["layers"], case["vocab"]
    body = L * sum(int(np.prod(_shape(case, s))) for s in SLOTS)
    head = V * H
    row_kv = 2 * L * nkv * hd * (2 if case["kv"] == "f16" else 4)  # one position's cache, all layers

    def forward(rows, start, heads=1):
        """Rows at [start, start + rows) in one forward: weights once, the cache before them once."""
        pairs = rows * start + rows * (rows + 1) / 2
        return ((body + head) * _per_weight(case) + row_kv * (start + rows) + 4 * H * rows + 4 * V * heads,
                2 * body * rows + 2 * head * heads + 4 * nq * hd * L * pairs)

    if case["kind"] in ("step", "prompt"):
        b, f = forward(case["rows"], case["start"])
        return {"bytes": b, "flops": f}
    if case["kind"] == "generate":
        parts = [forward(case["rows"], 0)] + [forward(1, case["rows"] + i) for i in range(case["steps"])]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    B, mean = case["batch"], (1 + case["rows"]) / 2
    b, f = forward(mean * B, 0, B)  # the prompts together, their caches apart
    f -= 4 * nq * hd * L * (mean * B * (mean * B + 1) / 2 - B * mean * (mean + 1) / 2)
    for i in range(case["steps"]):
        at = mean + i
        b += (body + head) * _per_weight(case) + B * (row_kv * (at + 1) + 4 * H + 4 * V)
        f += B * (2 * body + 2 * head + 4 * nq * hd * L * (at + 1))
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] == "linear":
        # exact block sums, then one f32 sum over the row's blocks
        return {"rel": 2e-6, "max": 2e-5}
    if case["order"] == "reference":
        return "exact"
    # Activations are rounded to 8 bits at every linear layer: where two correct
    # orders of a sum put a value on different sides of a rounding midpoint, the
    # code differs by one step, and the step travels on.  Between the two decode
    # orders, the same inputs give 1e-7 where no code differs, 1e-4 to 3e-3 (max
    # 6e-4 to 1e-2) on most rows and up to 2e-2 (max 0.07) on single rows and
    # with zero-mean codes.
    return {"rel": 3e-2, "max": 0.3, "differ": 0.0}


# ---- the same in 64 bits ------------------------------------------------------
def _q8_rows(x):
    """Q8_0 of f32 rows as the operator defines it: per block of 32 the scale amax/127 in f32, and each
    value times the scale's f32 reciprocal, rounded half away from zero."""
    b = x.reshape(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    p = (b * (1.0 / d)).double()
    q = torch.sign(p) * torch.floor(p.abs() + 0.5)
    return (q.clamp(-127, 127) * d.double()).reshape(x.shape)


def _rope(x, start):
    """Rotate-half RoPE of x [rows][heads][hd] at positions start.."""
    rows, _, hd = x.shape
    f = THETA ** (-2.0 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)
    a = (torch.arange(rows, device=x.device, dtype=torch.float64) + start)[:, None] * f
    c, s = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat((lo * c - hi * s, lo * s + hi * c), -1)


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _decoder(case, seed, sequences):
    """The decoder over token rows in 64 bits, with no 8-bit activations: per sequence (tokens, start) the
    logits of every row asked for. Each layer's matrices are made once for all sequences."""
    nq, nkv, hd, _ = WIDTHS[case["width"]]
    embed = _embedding(case, seed)
    xs = [embed[t.to(DEV).long()].double() for t, _, _ in sequences]
    head = _value(*_lm_head(case, seed, embed), case["weight"])
    del embed
    for layer in range(case["layers"]):
        W = {s: _value(*_linear(case, seed, layer, s), case["weight"]) for s in SLOTS}
        n0, n1 = (_norm(case, seed, layer, s) for s in (lh.N_INPUT, lh.N_POST))
        for i, (_, start, _) in enumerate(sequences):
            x = xs[i]
            rows = x.shape[0]
            a = _rms(x, n0)
            q = _rope((a @ W[lh.W_Q].T).reshape(rows, nq, hd), start)
            k = _rope((a @ W[lh.W_K].T).reshape(rows, nkv, hd), start).transpose(0, 1)
            v = (a @ W[lh.W_V].T).reshape(rows, nkv, hd).transpose(0, 1)
            if start:
                ck, cv = _cache(case, seed, layer)
                k, v = torch.cat((ck.double(), k), 1), torch.cat((cv.double(), v), 1)
            seen = torch.arange(start + rows, device=x.device)[None] <= torch.arange(rows, device=x.device)[:, None] + start
            ctx = torch.empty(rows, nq, hd, device=x.device, dtype=torch.float64)
            for h in range(nq):
                s = (q[:, h] @ k[h // (nq // nkv)].T / math.sqrt(hd)).masked_fill(~seen, -math.inf)
                ctx[:, h] = s.softmax(-1) @ v[h // (nq // nkv)]
            x = x + ctx.reshape(rows, -1) @ W[lh.W_O].T
            a = _rms(x, n1)
            gate = a @ W[lh.W_GATE].T
            xs[i] = x + (gate * gate.sigmoid() * (a @ W[lh.W_UP].T)) @ W[lh.W_DOWN].T
        del W
    w = _norm(case, seed, -1, 0)
    return [_rms(x[take], w) @ head.T for x, (_, _, take) in zip(xs, sequences)]


def exact(case, seed):
    if case["kind"] == "linear":
        g = _gen(seed, 1)
        codes = _codes(g, case["weight"], case["n"], case["k"])
        w = _value(codes, _scales(g, case["weight"], case["n"], case["k"]), case["weight"])
        return _q8_rows(_normal(_gen(seed, 6), case["rows"], case["k"])) @ w.T
    if case["sampled"]:
        return None  # which ids follow is the sampler's draw
    if case["kind"] in ("step", "prompt"):
        t = _tokens(case, seed)
        return {"logits": _decoder(case, seed, [(t, case["start"], slice(-1, None))])[0][0]}
    # The greedy loops' text counts on from the prompt's last token; each row's argmax has to say so.
    steps = case["steps"] - (case["kind"] == "generate")
    prompts = [_tokens(case, seed, s) for s in range(max(1, case["batch"]))]
    whole = [torch.cat((p, (int(p[-1]) + 1 + torch.arange(steps + 1)).remainder(case["vocab"]).to(torch.int32))) for p in prompts]
    # generate(): the row after the last token; a batch: the row that gave it
    cut = [w if case["kind"] == "generate" else w[:-1] for w in whole]
    out = _decoder(case, seed, [(c, 0, slice(p.numel() - 1, None)) for c, p in zip(cut, prompts)])
    for lg, p, w in zip(out, prompts, whole):
        said = w[p.numel():].to(lg.device).long()
        if not torch.equal(lg[: said.numel()].argmax(-1), said):
            raise AssertionError("the 64-bit greedy text is another one")
    if case["kind"] == "generate":
        return {"tokens": whole[0][prompts[0].numel():].numpy(), "logits": out[0][-1]}
    return {"tokens": np.concatenate([w.numpy() for w in whole]), "logits": torch.stack([lg[-1] for lg in out])}
