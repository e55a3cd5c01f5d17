"""Batched GEMV (M = 2..8) of every weight format at the edges of its launch
shapes: row tiles of 16 and their remainders, K of one slot, of odd slot
counts, and of partial slots where a format allows them (BF16 K % 8, Q4Mat
K % 32), K staged in one chunk, in several, and split over workgroups, and
outputs long enough for workgroups that walk several tile groups.

Reference: float64 products of the dequantized weights (the oracle's
decoders).  Bound, per row of y: Q4_K's activation limbs are within 2.5e-7 of
a block's absmax (q4k_mfma.hpp), those of Q4_0 and Q4Mat within 2^-30, and f32
sums round by 2^-24 a step, so each output is within 4e-7 * sum|w x|-like
terms; taken normwise over the output that is below 1e-5 at every size here,
the bound the single-row GEMVs are held to.
"""
import numpy as np
import pytest

from fresh_process import run_case
from helpers import GEMV_TOL, f32_to_bf16_rne, bf16_bits_to_f32, from_dev, normwise_err, say, to_dev

pytestmark = pytest.mark.gpu


def weights(rt, orc, fmt, rng, n, k):
    """(device bytes, float64 values) of a random weight in `fmt`."""
    if fmt == "q4mat":
        packed = rng.integers(0, 256, n * k // 2, dtype=np.uint8)
        scales = (0.002 + 0.004 * rng.random(n * k // 32)).astype(np.float32)
        nib = np.stack([packed & 15, packed >> 4], -1).reshape(-1).astype(np.int64)
        v = np.where(nib > 7, nib - 16, nib) * np.repeat(scales.astype(np.float64), 32)
        return rt.q4mat_upload(packed, scales, n, k), v.reshape(n, k)
    if fmt == "q4_0":
        b = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
        b[:, :2] = (0.002 + 0.004 * rng.random(b.shape[0])).astype(np.float16)[:, None].view(np.uint8)
        d = b[:, :2].copy().view(np.float16).astype(np.float64)
        q = np.concatenate([b[:, 2:] & 15, b[:, 2:] >> 4], 1).astype(np.float64) - 8
        return to_dev(b.reshape(-1)), (d * q).reshape(n, k)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    if fmt == "bf16":
        bits = f32_to_bf16_rne(w)
        return to_dev(bits), bf16_bits_to_f32(bits).astype(np.float64).reshape(n, k)
    blocks = orc.q4k_quantize(w)
    return to_dev(blocks), orc.q4k_dequant(blocks, n, k).astype(np.float64)


def run(rt, fmt, w, x, n, k):
    code = {"q4k": rt.Q4K, "bf16": rt.BF16, "q4_0": rt.Q4_0, "q4mat": rt.Q4MAT}[fmt]
    return from_dev(rt.gemv(code, w, to_dev(x), n, k))


SHAPES = [(1, 256, 2), (15, 512, 3), (17, 768, 4), (129, 1280, 5), (300, 2816, 8), (48, 12032, 4), (40, 8448, 7),
          (4112, 256, 8)]
TAILS = {"bf16": [(33, 8, 2), (70, 1160, 5)], "q4mat": [(33, 32, 2), (70, 1184, 5)]}


@pytest.mark.parametrize("fmt", ["q4k", "bf16", "q4_0", "q4mat"])
def test_batched_gemv_edges(rt, orc, fmt):
    for n, k, m in SHAPES + TAILS.get(fmt, []):
        say(f"[gemv batch {fmt}] {n} x {k}, M = {m}")
        rng = np.random.default_rng(n + k + m)
        w, v = weights(rt, orc, fmt, rng, n, k)
        x = rng.standard_normal((m, k)).astype(np.float32)
        x[-1] *= np.float32(1e-20)  # rows keep scales of their own
        y = run(rt, fmt, w, x, n, k)
        for r in range(m):
            want = v @ x[r].astype(np.float64)
            scale = np.abs(v) @ np.abs(x[r].astype(np.float64))
            assert np.max(np.abs(y[r] - want)) <= GEMV_TOL * np.max(scale), (fmt, n, k, m, r)
        assert np.array_equal(y, run(rt, fmt, w, x, n, k))  # the order of sums is fixed


@pytest.mark.parametrize("fmt", ["q4k", "q4_0", "q4mat"])
def test_batched_gemv_long_output(rt, orc, fmt):
    """Outputs of several rounds of workgroups: M = 8 (16-wave workgroups) and M = 3, rows checked throughout."""
    import torch
    n, k = 70001, 2560
    g = torch.Generator(device="cuda").manual_seed(3)
    rng = np.random.default_rng(3)
    base, v = weights(rt, orc, fmt, rng, 512, k)
    if fmt == "q4mat":  # the same 512 rows over and over: packed bytes, then scales
        off = rt.library().lib.rt_hip_q4mat_scales_offset(512, k)
        reps = -(-n // 512)
        pk, sc = base[:512 * k // 2].reshape(512, -1), base[off:off + 512 * k // 8].reshape(512, -1)
        buf = torch.zeros(rt.q4mat_bytes(n, k), dtype=torch.uint8, device="cuda")
        buf[:n * k // 2] = pk.repeat(reps, 1)[:n].reshape(-1)
        o = rt.library().lib.rt_hip_q4mat_scales_offset(n, k)
        buf[o:o + n * k // 8] = sc.repeat(reps, 1)[:n].reshape(-1)
        w = buf
    else:
        w = base.reshape(512, -1).repeat(-(-n // 512), 1)[:n].reshape(-1).contiguous()
    x = torch.randn((8, k), device="cuda", generator=g).cpu().numpy()
    for m in (3, 8):
        say(f"[gemv batch {fmt}] {n} x {k}, M = {m}")
        y = run(rt, fmt, w, x[:m], n, k)
        want = (x[:m].astype(np.float64) @ v.T)
        assert normwise_err(y[:, :512], want) <= GEMV_TOL
        for r0 in range(512, n, 512):  # every other copy of the rows gives the same sums
            r1 = min(n, r0 + 512)
            assert np.array_equal(y[:, r0:r1], y[:, :r1 - r0]), r0


def test_batched_gemv_without_workspace_room(rt):
    """A shape that is split over workgroups, captured without room to grow the
    workspace, keeps K inside its workgroups: accepted, and right."""
    say("[gemv batch] Q4_0 captured without workspace")
    run_case("gemv_q4_0")


@pytest.mark.parametrize("fmt", ["q4k", "bf16", "q4_0", "q4mat"])
def test_batched_gemv_nonfinite_rows(rt, orc, fmt):
    """One NaN or infinity in a row of x makes that row of y NaN or infinite,
    as an f32 sum with nonzero terms would, and leaves the other rows' bits."""
    n, k = 40, 768
    for m, bad in [(3, 1), (8, 6)]:
        rng = np.random.default_rng(m)
        w, _ = weights(rt, orc, fmt, rng, n, k)
        x = rng.standard_normal((m, k)).astype(np.float32)
        clean = run(rt, fmt, w, x, n, k)
        for value in (np.nan, np.inf, -np.inf):
            for at in (0, 421, k - 1):
                say(f"[gemv batch {fmt}] M = {m}, {value} at {at}")
                z = x.copy()
                z[bad, at] = value
                y = run(rt, fmt, w, z, n, k)
                assert not np.isfinite(y[bad]).any()
                if np.isnan(value):
                    assert np.isnan(y[bad]).all()
                assert np.array_equal(np.delete(y, bad, 0), np.delete(clean, bad, 0))


# rms error of ordinary rows against float64, relative to the result:
#  * f32 steps round by 2^-24 / sqrt(3) of their size, a random sum of s steps
#    grows as sqrt(s): over n steps 2^-24 / sqrt(3) * sqrt(n / 2).
#  * BF16: chains of half a chunk's 32-value steps, at most 100 steps a chunk.
#  * Q4_K: the blocks of 32, and the limbs' steps of 2^-20 where a block's
#    absmax is 2 to 4 (rms 2^-20 / sqrt(12)).
@pytest.mark.parametrize("fmt,n,k,m,steps,limbs", [("bf16", 12288, 12288, 8, 100, 0.0), ("bf16", 1024, 3072, 4, 96, 0.0),
                                                   ("q4k", 1024, 3072, 5, 96, 2.0 ** -20 / 12 ** 0.5),
                                                   ("q4k", 4096, 4096, 8, 128, 2.0 ** -20 / 12 ** 0.5)])
def test_batched_gemv_rounding(rt, fmt, n, k, m, steps, limbs):
    import torch
    say(f"[gemv batch rounding] {fmt} {n} x {k}, M = {m}")
    g = torch.Generator(device="cuda").manual_seed(n + m)
    w = torch.randn((n, k), device="cuda", generator=g) * 0.02
    if fmt == "bf16":
        code, data, v = rt.BF16, w.bfloat16().view(torch.int16), w.bfloat16()
    else:
        code, data = rt.Q4K, rt.quantize_q4k(w)
        v = rt.dequant_q4k(data, n, k).reshape(n, k)
    x = torch.randn((m, k), device="cuda", generator=g)
    y = rt.gemv(code, data, x, n, k).double()
    want = torch.cat([x.double() @ v[i:i + 2048].double().T.contiguous() for i in range(0, n, 2048)], 1)
    bound = (limbs ** 2 + (2.0 ** -24 / 3 ** 0.5) ** 2 * steps / 2) ** 0.5
    assert float((y - want).norm() / want.norm()) <= bound


@pytest.mark.parametrize("fmt,n,k,m", [("q4k", 16, 131072, 8), ("q4k", 256, 65536, 5), ("bf16", 40, 131072, 3),
                                       ("bf16", 256, 65536, 8), ("q4_0", 12288, 12288, 8), ("q4mat", 250, 35840, 7)])
def test_batched_gemv_long_k(rt, fmt, n, k, m):
    """K of many chunks: summed over workgroups, in up to 128 slices, and over
    more workgroups than the device holds at once (12288 x 12288); at most 4 times
    the time of a square of as many weights (kept inside few workgroups, up to 17)."""
    import torch
    say(f"[gemv batch long k] {fmt} {n} x {k}, M = {m}")
    gen = torch.Generator(device="cuda").manual_seed(k)

    def make(n, k):
        if fmt == "q4mat":
            off, w = rt.library().lib.rt_hip_q4mat_scales_offset(n, k), torch.empty(rt.q4mat_bytes(n, k), dtype=torch.uint8, device="cuda")
            w[:n * k // 2] = torch.randint(0, 256, (n * k // 2,), dtype=torch.uint8, device="cuda", generator=gen)
            w[off:off + n * k // 8] = (0.002 + 0.004 * torch.rand(n * k // 32, device="cuda", generator=gen)).view(torch.uint8)
            return rt.Q4MAT, w
        if fmt == "q4_0":
            b = torch.randint(0, 256, (n * k // 32, 18), dtype=torch.uint8, device="cuda", generator=gen)
            b[:, :2] = (0.002 + 0.004 * torch.rand(n * k // 32, device="cuda", generator=gen)).half()[:, None].view(torch.uint8)
            return rt.Q4_0, b.reshape(-1)
        w = torch.randn((n, k), device="cuda", generator=gen) * 0.02
        return (rt.BF16, w.bfloat16().view(torch.int16)) if fmt == "bf16" else (rt.Q4K, rt.quantize_q4k(w))

    def time_of(code, w, x, n, k):
        y, best = torch.empty((m, n), device="cuda"), 1e9
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                rt.gemv(code, w, x, n, k, y=y)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return y, best

    code, w = make(n, k)
    v = w.view(torch.bfloat16) if fmt == "bf16" else rt.dequant(code, w, n, k)
    x = torch.randn((m, k), device="cuda", generator=gen)
    y, t = time_of(code, w, x, n, k)
    want = torch.cat([x.double() @ v.reshape(n, k)[i:i + 2048].double().T.contiguous() for i in range(0, n, 2048)], 1)
    assert float((y.double() - want).abs().amax() / want.abs().amax()) <= GEMV_TOL
    side = max(1024, int((n * k) ** 0.5) // 256 * 256)
    code, w = make(side, side)
    assert t <= 4 * time_of(code, w, x[:, :side].contiguous(), side, side)[1]
