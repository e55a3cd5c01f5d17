"""The Q4_K quantizer at block counts that leave a wave's group of four blocks
partly empty, on values where a nibble's quotient sits next to a rounding
boundary, and on zeros, infinities, NaN and the ends of the f32 and f16
ranges: bytes equal to the oracle's."""
import numpy as np
import pytest

from helpers import say, to_dev

pytestmark = pytest.mark.gpu


def check(rt, orc, w, what):
    n, k = w.shape
    got = rt.quantize_q4k(to_dev(w)).cpu().numpy().reshape(-1, 144)
    want = np.asarray(orc.q4k_quantize(w), dtype=np.uint8).reshape(-1, 144)
    bad = np.flatnonzero((got != want).any(1))
    assert bad.size == 0, f"{what}: {bad.size} of {len(want)} blocks differ, first {bad[:4]}"


@pytest.mark.parametrize("n,k", [(1, 256), (1, 512), (3, 256), (1, 1024), (5, 256), (3, 1280), (17, 256), (7, 2304)])
def test_quantize_q4k_block_counts(rt, orc, n, k):
    say(f"[quantize blocks] {n} x {k}")
    rng = np.random.default_rng(n * 7 + k)
    check(rt, orc, (rng.standard_normal((n, k)) * 0.1).astype(np.float32), "normal")
    check(rt, orc, np.abs(rng.standard_normal((n, k))).astype(np.float32), "positive")


def test_quantize_q4k_near_boundaries(rt, orc):
    """Sums v + mn within 3 ulps of (i + 0.5) * scale: 63 steps of d give every
    scale a sub-block can have."""
    rng = np.random.default_rng(4)
    rows = []
    for d in (2.0 ** -24, 2.0 ** -14, 0.001, 0.0123, 1.0, 777.0):
        d = np.float32(np.float16(d))
        w = np.zeros((8, 8, 8, 32), np.float32)  # 8 rows of 8 blocks of 8 sub-blocks
        w[:] = (rng.integers(0, 15, w.shape) + 0.5) * (d * rng.integers(1, 64, (8, 8, 8, 1)))
        w[..., 0, 0] = d * np.float32(63 * 15)
        w = (w.view(np.int32) + rng.integers(-3, 4, w.shape)).astype(np.int32).view(np.float32)
        rows.append(w.reshape(8, 2048))
        neg = w - np.float32(d * 20)
        rows.append(neg.astype(np.float32).reshape(8, 2048))
    say("[quantize blocks] boundaries")
    check(rt, orc, np.concatenate(rows), "boundaries")


def test_quantize_q4k_special_values(rt, orc):
    rng = np.random.default_rng(5)
    w = rng.standard_normal((64, 1024)).astype(np.float32)
    special = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 1e-45, -1e-45, 1e-38, 3.4e38, -3.4e38, 1e5, -1e8, 7e6, 1e-7],
                       np.float32)
    at = rng.random(w.shape) < 0.003
    w[at] = rng.choice(special, at.sum())
    w[::7] = np.where(rng.random((len(w[::7]), 1024)) < 0.5, w[::7], 0.0)
    w[5], w[6], w[7] = 0.0, np.nan, -np.inf
    w[8, ::2], w[8, 1::2] = np.inf, -1.0
    w[9], w[10] = w[9] * np.float32(1e-40), w[10] * np.float32(1e36)
    w[11], w[12] = w[11] * np.float32(1e8), w[12] * np.float32(1e-7)
    say("[quantize blocks] special values")
    check(rt, orc, w, "special")
