"""Tokens into a call and logits out of it by kernels: odd vocabularies (a
logits row that ends inside a 16-byte store) and prompts around the kernels'
workgroup of 256."""
from dataclasses import replace

import numpy as np
import pytest

import oracle.oracle as orc
from alpaca_amd import synth
from alpaca_amd.model import HIPLlamaModel
from tests.helpers import assert_close, env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,prompt,persistent", [(1021, 1, 1), (1022, 1, 0), (1023, 255, 1), (1024, 256, 0),
                                                     (1025, 257, 1), (1026, 513, 0)])
def test_tokens_in_and_logits_out(hip_ctx, vocab, prompt, persistent):
    """The tolerance of the exact GEMM's model logits: 2e-3 absolute + 1e-3 relative, as in the smoke run."""
    spec = replace(synth.TINY, config=replace(synth.TINY.config, vocab_size=vocab))
    c = spec.config
    w = synth.build_weights(spec)
    cfg = dict(vocab=c.vocab_size, hidden=c.hidden_size, layers=c.layer_count, heads=c.head_count,
               kv_heads=c.kv_head_count, head_dim=c.head_dim, ffn=c.feed_forward_size, context=c.context_length,
               eps=c.rms_norm_eps, theta=c.rope_theta, interleaved=c.rope_interleaved)
    om = orc.OracleModel(cfg, {n: (t.dtype, t.data) for n, t in w.items()})
    kv = orc.OracleKV(cfg, prompt + 2, rounds_f16=True)
    tokens = np.random.default_rng(vocab).integers(0, vocab, prompt + 2).astype(np.int32)
    tokens[-1] = vocab - 1
    with env(ALPACA_HIP_PERSISTENT_DECODE=persistent):
        session = HIPLlamaModel(hip_ctx, c, w).make_session(capacity=prompt + 2, gemm_precision="exact")
    for part in (tokens[:prompt], tokens[prompt:prompt + 1], tokens[prompt + 1:]):
        assert_close(session.forward(part), orc.forward(om, kv, part), 2e-3, 1e-3, f"{vocab} after {len(part)}")
