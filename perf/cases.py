"""The workloads this library is measured by: what a program that runs Llama
models through it has it do, from a one-line message to a 4,096-token prompt,
single-token decode with a short and a long context, and token sampling.

A case is a dict of plain values:

``kind`` "generate": one session of a model whose weights are resident.  A pass
resets the session, appends a prompt (``forward``), then a second message if
``turn`` is set (``forward`` with the first one in the KV cache), then
``steps`` tokens one at a time (``decode``), and returns the logits of every
call.  The tokens are given, not taken from the logits, so that a rounding
difference cannot send two runs down different texts.

``kind`` "sample": ``draws`` tokens drawn from given logits, one after another
as a generation loop draws them.

The model shapes are the benchmark's (``alpaca_amd.synth``: C1 135M, C4 360M,
C5 1.7B).  ``layers`` is the depth; the 1.7B shape runs a block of its layers,
all of one size, so that its weights are made quickly.  Weights are random in
the named format, norm gains about 1, prompts uniform over the vocabulary.
"""
from __future__ import annotations

import functools
import math
from dataclasses import replace

import numpy as np
import torch

from alpaca_amd import synth
from alpaca_amd.model import HIPContext, HIPLlamaModel
from alpaca_amd.ops import HIPOps
from alpaca_amd.sampling import SplitMix64
from alpaca_amd.tensor import BY_NAME, QTensor

SHAPES = {"C1": synth.C1, "C4": synth.C4, "C5": synth.C5}
DEPTH = {"C1": 30, "C4": 32, "C5": 4}
WEIGHT_STD = 0.02  # of the projections, as in alpaca_amd.synth


def _generate(model, weights="q8_0", prompt=128, turn=0, steps=0, batch=512, precision="fast", kv="f16", layers=0):
    # batch 512 is make_session's default: longer prompts go in chunks of it
    return {"kind": "generate", "model": model, "layers": layers or DEPTH[model], "weights": weights, "prompt": prompt,
            "turn": turn, "steps": steps, "batch": batch, "precision": precision, "kv": kv}


def _sample(vocab, temperature, top_k, top_p, draws):
    return {"kind": "sample", "vocab": vocab, "temperature": temperature, "top_k": top_k, "top_p": top_p,
            "draws": draws}


def listed() -> list:
    def named(name, case):
        return dict(case, name=name)
    return [
        # A one-line message: the time to the first token, where launches and latency are all there is.
        named("message-11", _generate("C1", prompt=11)),
        # The reference's own short request: a 128-token prompt, then 16 tokens.
        named("request-128+16", _generate("C1", prompt=128, steps=16)),
        # Writing at length with a long context, the headline decode figure's setting.
        named("decode-at-2000", _generate("C1", prompt=2000, steps=48)),
        # The headline prefill: a 4,096-token prompt in one chunk.
        named("prefill-4096", _generate("C1", prompt=4096, batch=4096)),
        # A document of odd length through a session made with the defaults.
        named("prefill-1777-default", _generate("C1", prompt=1777)),
        # A document, then a question about it, 4-bit weights.
        named("q4-turn-1021+37", _generate("C4", "q4_0", prompt=1021, turn=37)),
        # An answer from the 4-bit model.
        named("q4-decode-300", _generate("C4", "q4_0", prompt=300, steps=24)),
        # Layers of a model large enough to fill the chip: a long prompt ...
        named("large-prefill-4096", _generate("C5", prompt=4096, batch=4096)),
        # ... and an ordinary one, then an answer.
        named("large-request-300+24", _generate("C5", prompt=300, steps=24)),
        # An unquantised model with the one-term activations.
        named("f16-prefill-700", _generate("C1", "f16", prompt=700, batch=1024, precision="fast-f16")),
        # The float32 mode with a float32 cache: the setting that numerics are checked against.
        named("exact-f32-150+4", _generate("C1", prompt=150, steps=4, precision="exact", kv="f32", layers=10)),
        # Drawing the next token with the usual sampler settings.
        named("sample-49152", _sample(49152, 0.8, 40, 0.95, 8)),
    ]


def _log_uniform(rng, lo, hi) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    r = rng.random()
    if r < 0.12:
        # plain temperature, top-k, top-p, or both
        k, p = rng.choice([(0, 1.0), (1, 1.0), (1, 0.0), (0, 0.0)])
        return _sample(_log_uniform(rng, 1000, 131072), round(rng.uniform(0.5, 1.3), 2),
                       _log_uniform(rng, 5, 300) if k else 0, p or round(rng.uniform(0.7, 0.98), 2),
                       rng.randint(4, 12))
    if r < 0.2:
        return _generate("C1", rng.choice(["q8_0", "q4_0", "f16"]), prompt=_log_uniform(rng, 2, 200),
                         steps=rng.randint(0, 4), precision="exact", kv=rng.choice(["f32", "f16"]),
                         layers=rng.randint(2, 10))
    model = rng.choice(["C1", "C1", "C4", "C5"])
    weights = rng.choice({"C1": ["q8_0", "q8_0", "f16"], "C4": ["q4_0", "q4_0", "q8_0"], "C5": ["q8_0"]}[model])
    longest = {"C1": 4096, "C4": 2500, "C5": 4096}[model]
    prompt = _log_uniform(rng, 16 if model == "C4" else 2, longest)
    what = rng.choice(["prefill", "prefill", "turn", "decode"])
    return _generate(model, weights, prompt=prompt,
                     turn=_log_uniform(rng, 2, 400) if what == "turn" else 0,
                     steps=rng.randint(2, 32) if what == "decode" else 0,
                     batch=rng.choice([512, 512, longest]),
                     precision=rng.choice(["fast", "fast", "fast", "fast-f16"]))


# ---------------------------------------------------------------- inputs

def _config(case):
    c = SHAPES[case["model"]].config
    return replace(c, layer_count=case["layers"])


def _positions(case) -> int:
    return case["prompt"] + case["turn"] + case["steps"]


def _blocks(g, rows, cols, fmt):
    """Raw bytes (GPU) of a random [rows, cols] matrix in ``fmt``."""
    v = torch.randn(rows, cols, generator=g, device="cuda") * WEIGHT_STD
    if fmt == "f16":
        return v.half().view(torch.uint8).reshape(-1)
    b = v.reshape(-1, 32)
    peak = b.gather(1, b.abs().argmax(1, keepdim=True))
    if fmt == "q8_0":
        d = peak.abs() / 127
        q = torch.round(b / d).clamp(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        d = peak / -8
        n = torch.floor(b / d + 8.5).clamp(0, 15).to(torch.uint8)
        q = n[:, :16] | (n[:, 16:] << 4)
    return torch.cat([d.half().view(torch.uint8), q], 1).reshape(-1)


def _tensors(case, seed):
    """(name, format, rows, cols, raw bytes on the GPU) of the case's weights."""
    c = _config(case)
    spec = replace(SHAPES[case["model"]], config=c)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for name in synth.tensor_names(spec):
        rows, cols = synth.tensor_shape(spec, name)
        if name.endswith("norm"):
            w = 1 + 0.1 * torch.randn(cols, generator=g, device="cuda")
            yield name, "f32", rows, cols, w.view(torch.uint8).reshape(-1)
        else:
            yield name, case["weights"], rows, cols, _blocks(g, rows, cols, case["weights"])


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, _config(case).vocab_size, _positions(case)).astype(np.int32)


def _logits(case, seed):
    # scale 3: a nucleus of some hundreds of tokens, as language models have
    return (np.random.default_rng(seed).standard_normal(case["vocab"]) * 3).astype(np.float32)


@functools.cache
def _context():
    return HIPContext(0)


def prepare(case, seed):
    if case["kind"] == "sample":
        rng = SplitMix64(seed)
        return {"case": case, "ops": HIPOps(_context()), "logits": _logits(case, seed),
                "u": [rng.uniform() for _ in range(case["draws"])]}
    weights = {n: QTensor(BY_NAME[f], r, c, raw.cpu().numpy()) for n, f, r, c, raw in _tensors(case, seed)}
    model = HIPLlamaModel(_context(), _config(case), weights)
    # the capacity is the default, the model's context length
    session = model.make_session(max_batch=case["batch"], kv_precision=case["kv"], gemm_precision=case["precision"])
    return {"case": case, "session": session, "tokens": _tokens(case, seed)}


def run(state):
    case = state["case"]
    if case["kind"] == "sample":
        return np.array([state["ops"].sample(state["logits"], case["temperature"], case["top_k"], case["top_p"], u)
                         for u in state["u"]])
    s, tokens = state["session"], state["tokens"]
    s.reset()
    p, t = case["prompt"], case["turn"]
    out = [s.forward(tokens[:p])]
    if t:
        out.append(s.forward(tokens[p:p + t]))
    for token in tokens[p + t:]:
        out.append(s.decode(token))
    return out


# ---------------------------------------------------------------- what a pass has to do

def work(case) -> dict:
    if case["kind"] == "sample":
        # each draw reads the logits; an exponential, a product and a sum for each
        return {"bytes": case["draws"] * 4 * case["vocab"], "flops": case["draws"] * 3 * case["vocab"]}
    c = _config(case)
    H, QW, KW, F, V, L = (c.hidden_size, c.query_width, c.kv_width, c.feed_forward_size, c.vocab_size, c.layer_count)
    per_weight = {"q8_0": 34 / 32, "q4_0": 18 / 32, "f16": 2}[case["weights"]]
    kv = 2 if case["kv"] == "f16" else 4
    layer = (QW + 2 * KW) * H + H * QW + 3 * H * F
    total_bytes, flops, pos = 0.0, 0.0, 0
    for n in [case["prompt"]] + ([case["turn"]] if case["turn"] else []) + [1] * case["steps"]:
        total_bytes += (L * layer + V * H) * per_weight + (2 * L + 1) * H * 4 + V * 4 + n * H * per_weight
        total_bytes += 2 * L * (pos + n) * KW * kv
        flops += 2 * n * L * layer + 2 * V * H
        flops += L * 4 * QW * (n * pos + n * (n + 1) / 2)
        pos += n
    return {"bytes": total_bytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    # About four times the measured distance from exact(): 4e-7 in float32 throughout; with the f16 cache, whose
    # rounding of K and V sets the rest, 3-6e-4 (two activation terms, or float32 ones) and up to 1e-3 (one term).
    if case["kv"] == "f32":
        return {"rel": 2e-6}
    return {"rel": 4e-3 if case["precision"] == "fast-f16" else 2e-3}


# ---------------------------------------------------------------- 64-bit result

def _dequantise(fmt, rows, cols, raw):
    if fmt == "f32":
        return raw.view(torch.float32).double().reshape(rows, cols)
    if fmt == "f16":
        return raw.view(torch.float16).double().reshape(rows, cols)
    b = raw.reshape(-1, 34 if fmt == "q8_0" else 18)
    d = b[:, :2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        q = b[:, 2:].contiguous().view(torch.int8).double()
    else:
        n = b[:, 2:].to(torch.int32)
        q = torch.cat([n & 15, n >> 4], 1).double() - 8
    return (d * q).reshape(rows, cols)


def _norm(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def exact(case, seed):
    if case["kind"] == "sample":
        return None
    c = _config(case)
    hd, groups = c.head_dim, c.head_count // c.kv_head_count
    w = {n: (f, r, k, raw) for n, f, r, k, raw in _tensors(case, seed)}
    tokens = torch.from_numpy(_tokens(case, seed)).long().cuda()
    T = len(tokens)
    embed = _dequantise(*w["token_embd"])
    x = embed[tokens]
    freq = c.rope_theta ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * freq
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(v):
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    causal = torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)
    for li in range(c.layer_count):
        m = {n: _dequantise(*w[f"blk.{li}.{n}"]) for n in synth.LAYER_TENSORS}
        h = _norm(x, m["attn_norm"], c.rms_norm_eps)
        q = rope((h @ m["attn_q"].T).reshape(T, -1, hd))
        k = rope((h @ m["attn_k"].T).reshape(T, -1, hd))
        v = (h @ m["attn_v"].T).reshape(T, -1, hd)
        heads = []
        for i in range(c.head_count):
            s = (q[:, i] @ k[:, i // groups].T) / math.sqrt(hd)
            heads.append(torch.softmax(s.masked_fill_(causal, -math.inf), -1) @ v[:, i // groups])
        x = x + torch.cat(heads, 1) @ m["attn_output"].T
        h = _norm(x, m["ffn_norm"], c.rms_norm_eps)
        x = x + (torch.nn.functional.silu(h @ m["ffn_gate"].T) * (h @ m["ffn_up"].T)) @ m["ffn_down"].T
    ends = [case["prompt"]] + ([case["prompt"] + case["turn"]] if case["turn"] else [])
    ends += range(ends[-1] + 1, T + 1)
    rows = _norm(x[[e - 1 for e in ends]], _dequantise(*w["output_norm"]), c.rms_norm_eps)
    return list((rows @ embed.T).unbind(0))
