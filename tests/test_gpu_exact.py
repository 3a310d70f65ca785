"""The float32 kernels of the exact mode: the GEMMs, whose workgroups' waves take
a 32-weight block each or, on full grids, 64x64 tiles (bit for bit the CPU
reference's sums), and the attention of several queries on the float32 matrix
instructions.
"""
import numpy as np
import pytest

import oracle.oracle as orc
from alpaca_amd.tensor import F16, Q4_0, Q8_0, encode
from tests.helpers import assert_close
from tests.test_gpu_kernels import FORMATS, _f16, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(2, 70, 32), (3, 64, 544), (16, 65, 512), (150, 960, 576), (300, 130, 2560),
                                   (37, 200, 8192), (520, 64, 96)])
@pytest.mark.parametrize("name,dt", FORMATS)
def test_exact_gemm_bits(hip_ops, name, dt, m, n, k):
    """One block a row, a last phase with fewer blocks than waves (17 over 9), many phases (256
    blocks), one, two and four rows a lane, partial row and column groups: the CPU reference's
    float32 results bit for bit in the store and residual epilogues; SwiGLU within the exact
    GEMM's tolerance (expf differs from the host's in the last bit)."""
    x, res = rand((m, k), 700 + m), rand((m, n), 701, 5)
    w, wu = encode(rand((n, k), 702, 0.3), dt), encode(rand((n, k), 703, 0.3), dt)
    y, u = orc.linear(x, dt, w.data, n), orc.linear(x, dt, wu.data, n)
    for what, got, want in (("store", hip_ops.linear(x, w, "exact"), y),
                            ("residual", hip_ops.linear_add(x, w, res, "exact"), orc.add(res, y))):
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{name} {what}"
    assert_close(hip_ops.gate_up_silu(x, w, wu, "exact"), orc.mul(orc.silu(y), u), 2e-4, 1e-4, f"{name} swiglu")


@pytest.mark.parametrize("name,dt,m,n,k", [("Q8_0", Q8_0, 1061, 1490, 96), ("Q4_0", Q4_0, 1061, 640, 544),
                                           ("F16", F16, 1301, 1800, 64), ("Q8_0", Q8_0, 25000, 65, 32)])
def test_exact_gemm_bits_on_full_grids(hip_ops, name, dt, m, n, k):
    """Outputs past the 64x64 tiles' share of a 256-CU chip (1.5, 0.62 and 2.2 tiles a CU), partial
    tiles in both directions: bit for bit as in test_exact_gemm_bits."""
    x, res = rand((m, k), 720, 1), rand((m, n), 721, 5)
    w, wu = encode(rand((n, k), 722, 0.3), dt), encode(rand((n, k), 723, 0.3), dt)
    y, u = orc.linear(x, dt, w.data, n), orc.linear(x, dt, wu.data, n)
    for what, got, want in (("store", hip_ops.linear(x, w, "exact"), y),
                            ("residual", hip_ops.linear_add(x, w, res, "exact"), orc.add(res, y))):
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{name} {what}"
    assert_close(hip_ops.gate_up_silu(x, w, wu, "exact"), orc.mul(orc.silu(y), u), 2e-4, 1e-4, f"{name} swiglu")


@pytest.mark.parametrize("tokens,start,heads,kv,hd", [(2, 0, 4, 2, 32), (15, 1, 9, 3, 64), (16, 48, 9, 3, 64),
                                                      (17, 1000, 15, 5, 64), (150, 0, 9, 3, 64), (33, 31, 4, 4, 96),
                                                      (40, 77, 8, 2, 128), (20, 5, 4, 2, 160), (9, 100, 2, 1, 256)])
def test_float32_attention_of_several_queries(hip_ops, tokens, start, heads, kv, hd):
    """Partial query and key tiles, waves without a key tile, head dims of the tiled kernel and past
    it: the tolerances of the single-query kernels (test_attention_causal_gqa)."""
    cap = start + tokens + 3
    q, k, v = rand((tokens, heads, hd), 801), rand((cap, kv, hd), 802), rand((cap, kv, hd), 803)
    assert_close(hip_ops.attention(q, k, v, start, "f32"), orc.attention(q, k, v, start), 2e-6, 1e-5, "f32 cache")
    assert_close(hip_ops.attention(q, k, v, start, "f16"), orc.attention(q, _f16(k), _f16(v), start), 2e-5, 1e-4,
                 "f16 cache")


@pytest.mark.parametrize("tokens,start,heads,kv,hd", [(2, 126, 9, 3, 64), (2, 127, 9, 3, 64), (11, 1013, 32, 32, 64),
                                                      (15, 300, 4, 2, 32), (9, 2000, 8, 2, 128), (13, 131, 4, 4, 96),
                                                      (20, 600, 32, 8, 64), (33, 600, 32, 8, 64)])
def test_float32_attention_of_few_queries_over_many_keys(hip_ops, tokens, start, heads, kv, hd):
    """Both sides of the rules for eight or sixteen waves a workgroup (128 keys, 64 workgroups): the
    tolerances of test_float32_attention_of_several_queries."""
    cap = start + tokens + 3
    q, k, v = rand((tokens, heads, hd), 821), rand((cap, kv, hd), 822), rand((cap, kv, hd), 823)
    assert_close(hip_ops.attention(q, k, v, start, "f32"), orc.attention(q, k, v, start), 2e-6, 1e-5, "f32 cache")
    assert_close(hip_ops.attention(q, k, v, start, "f16"), orc.attention(q, _f16(k), _f16(v), start), 2e-5, 1e-4,
                 "f16 cache")


@pytest.mark.parametrize("tokens,start,hd", [(20, 0, 64), (16, 37, 32), (37, 5, 128)])
def test_float32_attention_keeps_later_values_from_earlier_queries(hip_ops, tokens, start, hd):
    """A value that is an infinity or NaN reaches the queries that see its key and no others."""
    cap = start + tokens
    q, k, v = rand((tokens, 4, hd), 811), rand((cap, 2, hd), 812), rand((cap, 2, hd), 813)
    v[start + 9, 0, 3], v[start + tokens - 2, 1, hd - 1] = np.inf, np.nan
    got, want = hip_ops.attention(q, k, v, start, "f32"), orc.attention(q, k, v, start)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    seen = np.isfinite(want)
    assert_close(got[seen], want[seen], 2e-6, 1e-5, "finite outputs")


@pytest.mark.parametrize("cache", ["f32", "f16"])
@pytest.mark.parametrize("tokens,start,hd", [(11, 0, 64), (11, 150, 64), (15, 401, 128)])
def test_few_queries_do_not_see_later_values(hip_ops, tokens, start, hd, cache):
    """The same for calls of 2 to 15 tokens, over both caches and with four, eight and sixteen waves."""
    cap = start + tokens
    q, k, v = rand((tokens, 4, hd), 831), rand((cap, 2, hd), 832), rand((cap, 2, hd), 833)
    v[start + 4, 0, 3], v[start + tokens - 2, 1, hd - 1] = np.inf, np.nan
    got = hip_ops.attention(q, k, v, start, cache)
    want = orc.attention(q, k, v, start) if cache == "f32" else orc.attention(q, _f16(k), _f16(v), start)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    seen = np.isfinite(want)
    assert_close(got[seen], want[seen], *((2e-6, 1e-5) if cache == "f32" else (2e-5, 1e-4)), "finite outputs")
