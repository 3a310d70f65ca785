"""The prefill GEMM for few rows (kernels_gemm_small.hip): K split over a
workgroup's waves, the smallest of four tiles whose grid is at most one
workgroup per CU, the RMSNorm inside the kernel on the two smallest.

Against the oracle at the shapes where each tile is chosen, with partial tiles
in both directions, and against the pipelined tiles (ALPACA_HIP_GEMM_TILE
forces one, read per launch) through sessions, where the same float32 products
are summed in another order: 1e-5 of the logit peak, as between the pipelined
tiles and their two-K-set form.  (Calls of 2 to 15 tokens have no pipelined form:
there the override changes nothing, and what they are held to is the float32
kernels, here and in test_gpu_few_rows.)
"""
from dataclasses import replace

import numpy as np
import pytest

import oracle.oracle as orc
from alpaca_amd import synth
from alpaca_amd.model import HIPLlamaModel
from alpaca_amd.tensor import F16, Q4_0, Q8_0, encode
from tests.helpers import env
from tests.test_gpu_kernels import FORMATS, rand
from tests.test_gpu_model import built

pytestmark = pytest.mark.gpu

# (rows, N, K): 16x16, 16x32, 32x32 and 32x64 tiles, then past one workgroup per CU (256)
SHAPES = [(16, 200, 576), (33, 1000, 64), (100, 960, 576), (250, 968, 1536), (500, 1000, 2560), (512, 1600, 960)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("name,dt", FORMATS)
def test_small_tiles_against_the_oracle(hip_ops, name, dt, m, n, k):
    """Store, residual and SwiGLU epilogues: two activation terms within the exact GEMM's tolerance
    2e-4 + 1e-4 |y|; one term within its input rounding, 2^-10 * sum |x w| (each x off by at most
    2^-11 relative, and as much again for float32 sums), on the store."""
    x = rand((m, k), 9000 + m)
    w, wu = encode(rand((n, k), 9100 + n, 0.3), dt), encode(rand((n, k), 9200 + n, 0.3), dt)
    res = rand((m, n), 9300, 5)
    y, u = orc.linear(x, dt, w.data, n), orc.linear(x, dt, wu.data, n)
    for what, got, want in (("store", hip_ops.linear(x, w, "fast"), y),
                            ("residual", hip_ops.linear_add(x, w, res, "fast"), orc.add(res, y)),
                            ("swiglu", hip_ops.gate_up_silu(x, w, wu, "fast"), orc.mul(orc.silu(y), u))):
        err, tol = np.abs(got.astype(np.float64) - want), 2e-4 + 1e-4 * np.abs(want)
        assert (err <= tol).all(), f"{name} {what}: worst error / tolerance {(err / tol).max():.3f}"
    deq = np.abs(orc.dequantize(dt, w.data, n * k).reshape(n, k)).astype(np.float64)
    err = np.abs(hip_ops.linear(x, w, "fast-f16").astype(np.float64) - y)
    bound = 2.0**-10 * (np.abs(x).astype(np.float64) @ deq.T) + 1e-5
    assert (err <= bound).all(), f"{name} one term: worst error / bound {(err / bound).max():.3f}"


def shaped(spec, name, dtype=None, **cfg):
    s = replace(spec, config=replace(spec.config, layer_count=2, vocab_size=2048, context_length=1100, **cfg), name=name)
    return s if dtype is None else replace(s, dtype=dtype)


SPECS = [shaped(synth.C1, "c1-shape"), shaped(synth.C1, "c1-shape-f16", F16), shaped(synth.C4, "c4-shape", Q4_0),
         shaped(synth.C1, "hd128", Q8_0, head_count=8, kv_head_count=2, head_dim=128)]


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("spec", SPECS, ids=lambda s: s.name)
def test_sessions_match_the_pipelined_tiles(hip_ctx, spec, kv):
    """Prompts of 2 to 700 tokens (the RMSNorm in the GEMM and before it, the RoPE epilogue at a
    non-zero position in the second call), second terms on every row, and a decode step over the
    cache they wrote.  With a float32 cache only the order of float32 sums differs: 1e-5 of the
    logit peak.  With the f16 cache a K or V element whose sum differs in its last bit can round to
    the neighbouring f16, 2^-11 of its value, which over two or three cached rows is one of the few
    terms of a head's output: half of 2^-11 of the peak (2.5e-4), as for two-stream prefills; below
    16 rows those calls are also held to the float32 kernels (ALPACA_HIP_PREFILL_GEMM=f32) by it."""
    tol = 1e-5 if kv == "f32" else 2.5e-4
    model = HIPLlamaModel(hip_ctx, spec.config, built(spec))
    prompt = synth.prompt_tokens(spec, 1000)
    with env(ALPACA_HIP_LO_ROWS="all"):
        a = model.make_session(max_batch=700, kv_precision=kv)
        b = model.make_session(max_batch=700, kv_precision=kv)
    with env(ALPACA_HIP_PREFILL_GEMM="f32"):
        f32 = model.make_session(max_batch=700, kv_precision=kv)
    for n in (2, 15, 16, 17, 37, 64, 130, 257, 300, 511, 700):
        for s in (a, b, f32):
            s.reset()
        for chunk in (prompt[:n], prompt[n:n + 9], prompt[n + 9:n + 10]):
            got = a.forward(chunk)
            with env(ALPACA_HIP_GEMM_TILE="64x64"):
                want = b.forward(chunk)
            peak = float(np.abs(want).max())
            d = float(np.abs(got - want).max())
            print(f"[metrics] {spec.name} {kv} n={n}+{len(chunk)}: small against pipelined max |d| {d / peak:.2e} of the peak")
            assert d <= tol * peak, f"{spec.name} {kv} n={n} chunk {len(chunk)}: {d / peak:.2e} of the peak"
            if n < 16:
                d = float(np.abs(got - f32.forward(chunk)).max())
                assert d <= tol * peak, f"{spec.name} {kv} n={n} against float32: {d / peak:.2e} of the peak"
    model.close()
