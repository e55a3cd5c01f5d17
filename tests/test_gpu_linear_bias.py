"""rt_hip_linear_forward with a bias against the same call without one, plus
the bias: one f32 addition per output, so the bits are the same whether the
GEMV's kernel adds it (Q4_K at any M, the other formats at M = 2..8) or a
second launch does.  Sizes: row tiles of 16 and their remainders, K held in
registers while staged and K past that (the M = 1 kernel's remainder loop),
outputs of several workgroup rounds, and K split over workgroups.
"""
import numpy as np
import pytest

from helpers import f32_to_bf16_rne, from_dev, say, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [(1, 256), (15, 512), (33, 768), (129, 3072), (300, 11264), (3072, 1024), (5000, 2816), (9000, 9216)]


def weight(rt, fmt, rng, n, k):
    if fmt == "q4mat":
        packed = rng.integers(0, 256, n * k // 2, dtype=np.uint8)
        return rt.Q4MAT, rt.q4mat_upload(packed, np.full(n * k // 32, 0.003, np.float32), n, k)
    if fmt == "q4_0":
        b = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
        b[:, :2] = np.float16(0.003).reshape(1).view(np.uint8)
        return rt.Q4_0, to_dev(b.reshape(-1))
    w = rng.standard_normal((n, k)).astype(np.float32) * np.float32(0.02)
    return (rt.BF16, to_dev(f32_to_bf16_rne(w))) if fmt == "bf16" else (rt.Q4K, rt.quantize_q4k(to_dev(w)))


@pytest.mark.parametrize("fmt", ["q4k", "bf16", "q4_0", "q4mat"])
def test_bias_is_one_addition(rt, fmt):
    import torch
    for n, k in SHAPES:
        rng = np.random.default_rng(n + k)
        code, w = weight(rt, fmt, rng, n, k)
        bias = rng.standard_normal(n).astype(np.float32)
        for m in (1, 2, 5, 8):
            say(f"[linear bias {fmt}] {n} x {k}, M = {m}")
            x = to_dev(rng.standard_normal((m, k)).astype(np.float32))
            plain = from_dev(rt.linear_forward(code, w, x, n, k))
            guard = torch.full((m * n + 64,), 7.0, device="cuda")
            y = guard[:m * n].view(m, n)
            rt.linear_forward(code, w, x, n, k, bias=to_dev(bias), y=y)
            assert np.array_equal(from_dev(y), plain + bias), (n, k, m)
            assert (from_dev(guard)[m * n:] == 7.0).all()
