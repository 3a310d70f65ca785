"""Calls of 2 to 15 tokens of the fast modes: short messages, and what is left of
a prompt past its last whole chunk.
"""
from dataclasses import replace

import numpy as np
import pytest

import oracle.oracle as orc
from alpaca_amd import synth
from alpaca_amd.model import HIPLlamaModel
from alpaca_amd.tensor import F16, encode
from tests.helpers import assert_close
from tests.test_gpu_model import built

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
