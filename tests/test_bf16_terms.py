"""The split of float32 activations and f16 weights into bf16 terms that the
few-row GEMM multiplies (csrc/kernels_gemm_small.hip bf16_split), restated in numpy."""
import numpy as np


def terms(x, n):
    out = []
    for _ in range(n):
        t = (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
        out.append(t)
        x = (x - t).astype(np.float32)
    return out, x


def test_three_terms_hold_a_float32():
    bits = np.random.default_rng(0).integers(0, 2**32, 4_000_000, dtype=np.uint64).astype(np.uint32)
    edges = np.array([0, 1, 0xFFFF, 0x10000, 0x7FFFFF], np.uint32)
    exps = (np.arange(25, 255, dtype=np.uint32)[:, None] << 23) | edges
    x = np.concatenate([bits, exps.ravel(), (exps | np.uint32(1 << 31)).ravel()]).view(np.float32)
    x = x[np.isfinite(x) & (np.abs(x) >= 2.0**-102)]
    parts, left = terms(x, 3)
    assert not left.any()
    assert np.array_equal(sum(p.astype(np.float64) for p in parts), x.astype(np.float64))
    assert all(((p == 0) | (np.abs(p) >= 2.0**-126)).all() for p in parts)


def test_two_terms_hold_an_f16_and_one_a_quant():
    h = np.arange(65536, dtype=np.uint16).view(np.float16).astype(np.float32)
    parts, left = terms(h[np.isfinite(h)], 2)
    assert not left.any()
    q = np.arange(-128, 128).astype(np.float32)
    assert not terms(q, 1)[1].any()
