"""Calls of 2 to 15 tokens of the fast modes: short messages, and what is left of
a prompt past its last whole chunk.
"""
from dataclasses import replace

import numpy as np
import pytest

import oracle.oracle as orc
from alpaca_amd import synth
from alpaca_amd.model import HIPLlamaModel
from alpaca_amd.tensor import F16, F32, Q4_0, Q8_0, encode
from tests.helpers import assert_close, env
from tests.test_gpu_kernels import FORMATS
from tests.test_gpu_model import built, oracle_cfg

pytestmark = pytest.mark.gpu

SPEC = replace(synth.C1, config=replace(synth.C1.config, layer_count=2, vocab_size=2048, context_length=256),
               name="few-rows")


@pytest.mark.parametrize("precision", ["fast", "fast-f16"])
def test_short_calls_use_the_quantised_weights(hip_ctx, precision):
    """The prefill weight cache holds f16 roundings of the weights (2^-11 of each), for prompts of 16
    tokens and more; shorter calls read the quants, so a model with the cache gives the same bits."""
    w = built(SPEC)
    models = [HIPLlamaModel(hip_ctx, SPEC.config, w, prefill_weight_cache=cache) for cache in (True, False)]
    a, b = (m.make_session(gemm_precision=precision) for m in models)
    prompt = synth.prompt_tokens(SPEC, 40)
    for part in (prompt[:11], prompt[11:26], prompt[26:28], prompt[28:29]):
        assert np.array_equal(a.forward(part).view(np.uint32), b.forward(part).view(np.uint32)), len(part)
    for m in models:
        m.close()


@pytest.mark.parametrize("hd", [64, 128])
def test_short_calls_keep_queries_past_the_f16_range(hip_ctx, hd):
    """Queries around 2^17 (past 65,504) against keys around 2^-13: scores of a few units, finite in
    float32.  Against the exact mode, whose GEMMs sum in another order, so that a cached key can round
    to the neighbouring f16: 2^-11 of a score of up to about 30, an eighth of the values' differences
    at the softmax, 1e-2 of the logit peak."""
    spec = replace(SPEC, dtype=F16, name=f"large-queries-{hd}",
                   config=replace(SPEC.config, head_dim=hd, head_count=9 if hd == 64 else 3,
                                  kv_head_count=3 if hd == 64 else 1))
    w = dict(built(spec))
    for li in range(spec.config.layer_count):
        for name, scale in (("attn_q", 2.0**18), ("attn_k", 2.0**-13)):
            t = w[f"blk.{li}.{name}"]
            v = orc.dequantize(t.dtype, t.data, t.rows * t.cols).reshape(t.rows, t.cols)
            w[f"blk.{li}.{name}"] = encode(v * np.float32(scale), F16)
    model = HIPLlamaModel(hip_ctx, spec.config, w)
    fast, exact = (model.make_session(gemm_precision=p) for p in ("fast", "exact"))
    prompt = synth.prompt_tokens(spec, 40)
    for part in (prompt[:11], prompt[11:26], prompt[26:28]):
        want = exact.forward(part)
        assert np.isfinite(want).all()
        assert_close(fast.forward(part), want, 1e-2 * float(np.abs(want).max()), 0.0, f"{len(part)} tokens")
    model.close()


# One layer whose attention adds nothing (the value projection is zero), so that the f16 cache's
# rounding leaves the logits alone and what remains is the FFN and the head.
def ffn_model(hip_ctx, dtype, gain, up, down):
    spec = replace(SPEC, dtype=dtype, config=replace(SPEC.config, layer_count=1), name=f"ffn-only-{dtype}")
    c = spec.config
    w = dict(built(spec))

    def scaled(name, by):
        t = w[name]
        v = orc.dequantize(t.dtype, t.data, t.rows * t.cols).reshape(t.rows, t.cols)
        w[name] = encode((v * np.float32(by)).astype(np.float32), dtype)
    for name, by in (("blk.0.attn_v", 0.0), ("blk.0.ffn_up", up), ("blk.0.ffn_down", down)):
        scaled(name, by)
    w["blk.0.ffn_norm"] = encode(np.full((1, c.hidden_size), gain, np.float32), F32)
    cfg = oracle_cfg(c)
    return HIPLlamaModel(hip_ctx, c, w), orc.OracleModel(cfg, {n: (t.dtype, t.data) for n, t in w.items()}), cfg


# (FFN norm gain, scale of up, of down): what the few-row GEMMs read
MAGNITUDES = {
    "ordinary": (1.0, 1.0, 1.0),
    # normalised rows around 1e-3: an f16 pair holds 15 of their 24 bits
    "small rows": (2.0**-10, 2.0**10, 2.0**10),
    # SwiGLU products around 1e-6, in the subnormals of f16
    "small products": (2.0**-7, 2.0**-3, 2.0**18),
    # products past 65,504, which f16 terms turn into infinities and their sums into NaN
    "large products": (1.0, 2.0**18, 1.0),
}


@pytest.mark.parametrize("name,dt", FORMATS)
@pytest.mark.parametrize("what", list(MAGNITUDES))
def test_short_calls_keep_float32_activations(hip_ctx, name, dt, what):
    """2, 11 and 15 tokens against the oracle, whose sums are float32 too: each of the three GEMMs in
    the logits' path sums up to 1,536 products, 2^-24 times a few tens of the terms' root mean square
    in either order, and the norms and SiLU a few 2^-23 more: 4e-6 of the logit peak."""
    model, om, cfg = ffn_model(hip_ctx, dt, *MAGNITUDES[what])
    tokens = synth.prompt_tokens(SPEC, 15)
    for precision in ("fast", "fast-f16"):
        for n in (2, 11, 15):
            got = model.make_session(gemm_precision=precision).forward(tokens[:n])
            want = orc.forward(om, orc.OracleKV(cfg, 20, rounds_f16=True), tokens[:n])
            assert_close(got, want, 4e-6 * float(np.abs(want).max()), 0.0, f"{name} {what} {precision} {n}")
    model.close()


# (hidden, heads, KV heads, head dim, FFN): K not a multiple of a stage's 64 (the float32 GEMM takes
# those), norms inside the GEMM and before it (hidden past 1,024), 16x32 tiles past one workgroup
# a CU (FFN past 8,192), head dims without the flash kernel (32, 96, 160)
FORMS = [(96, 3, 1, 32, 160), (192, 4, 2, 96, 256), (320, 2, 2, 160, 320), (1088, 4, 1, 128, 512),
         (512, 8, 4, 64, 8256), (2048, 32, 32, 64, 1024)]


@pytest.mark.parametrize("dt", [Q8_0, Q4_0, F16])
@pytest.mark.parametrize("hidden,heads,kv,hd,ffn", FORMS)
def test_short_calls_of_every_form(hip_ctx, hidden, heads, kv, hd, ffn, dt):
    """Two calls, the second over the cache of the first, against the exact mode: sums in another
    order, so a K or V element can round to the neighbouring f16, and half of 2^-11 of the logit peak
    as in test_gpu_small_gemm."""
    spec = replace(SPEC, dtype=dt, name="form", config=replace(
        SPEC.config, layer_count=2, hidden_size=hidden, head_count=heads, kv_head_count=kv, head_dim=hd,
        feed_forward_size=ffn, vocab_size=512))
    model = HIPLlamaModel(hip_ctx, spec.config, built(spec))
    fast, exact = (model.make_session(gemm_precision=p) for p in ("fast", "exact"))
    tokens = synth.prompt_tokens(spec, 40)
    for part in (tokens[:2], tokens[2:13], tokens[13:28], tokens[28:33]):
        want = exact.forward(part)
        assert_close(fast.forward(part), want, 2.5e-4 * float(np.abs(want).max()), 0.0, f"{len(part)} tokens")
    model.close()


@pytest.mark.parametrize("hd", [32, 64, 128])
def test_short_calls_rotate_and_append_as_the_separate_kernel(hip_ctx, hd):
    """RoPE and the KV append in the GEMM's epilogue against the GEMM and then the RoPE kernel: the same
    products and roundings, so the same bits, in the logits and in the decode step over the cache."""
    spec = replace(SPEC, name=f"rope-{hd}", config=replace(SPEC.config, head_dim=hd, head_count=4, kv_head_count=2))
    model = HIPLlamaModel(hip_ctx, spec.config, built(spec))
    fused = model.make_session()
    with env(ALPACA_HIP_FUSE_QKV_ROPE=0):
        apart = model.make_session()
    tokens = synth.prompt_tokens(spec, 40)
    for part in (tokens[:15], tokens[15:17], tokens[17:28], tokens[28:29]):
        assert np.array_equal(fused.forward(part).view(np.uint32), apart.forward(part).view(np.uint32)), len(part)
    model.close()
