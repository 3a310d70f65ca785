"""Calls of 2 to 15 tokens of the fast modes: short messages, and what is left of
a prompt past its last whole chunk.
"""
from dataclasses import replace

import numpy as np
import pytest

from alpaca_amd import synth
from alpaca_amd.model import HIPLlamaModel
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
