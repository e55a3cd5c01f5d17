"""FLUX's attention at the edges of its blocks and at values its bf16 limbs do
not take: 128- and 256-query blocks, 32-key tiles and every padded head width;
values past 2^64 (2^48 in v, 2^55 in q), infinities and NaN, which go through f32
matrix steps; products that overflow; tiny values; a capture without workspace.

Bound: FLUX_ATTN_TOL of test_gpu_flux_attention.py (1e-5 of the largest
output) against float64."""
import numpy as np
import pytest

from fresh_process import run_case
from helpers import from_dev, normwise_err, say, to_dev

pytestmark = pytest.mark.gpu

FLUX_ATTN_TOL = 1e-5


def exact(q, k, v, h, d):
    """float64 attention; inputs as f32 arithmetic sees them, so a score past
    the f32 range is infinite."""
    t = q.shape[0]
    q, k, v = (a.astype(np.float64).reshape(t, h, d).transpose(1, 0, 2) for a in (q, k, v))
    with np.errstate(all="ignore"):
        s = (q @ k.transpose(0, 2, 1))
        s = np.where(np.abs(s) > np.finfo(np.float32).max, np.sign(s) * np.inf, s) / np.sqrt(d)
        w = np.exp(s - s.max(-1, keepdims=True))
        w = w / w.sum(-1, keepdims=True)
        w = np.where(w < 1e-45, 0.0, w)
        out = w @ v
    return out.transpose(1, 0, 2).reshape(t, h * d)


def run(rt, q, k, v, h, d):
    return from_dev(rt.flux_attention(to_dev(q), to_dev(k), to_dev(v), h, d))


def rand(t, h, d):
    rng = np.random.default_rng(t * 31 + h * 5 + d)
    return [rng.standard_normal((t, h * d)).astype(np.float32) for _ in range(3)]


@pytest.mark.parametrize("t,h,d", [(31, 2, 32), (33, 1, 40), (96, 3, 128), (128, 2, 64), (129, 260, 8), (255, 200, 16),
                                   (257, 130, 40), (513, 90, 64), (520, 100, 72), (800, 70, 128), (100, 300, 120)])
def test_flux_attention_block_edges(rt, t, h, d):
    say(f"[flux limbs] t={t} heads={h} head_dim={d}")
    q, k, v = rand(t, h, d)
    got, want = run(rt, q, k, v, h, d), exact(q, k, v, h, d)
    assert normwise_err(got, want) <= FLUX_ATTN_TOL
    for hh in range(0, h, 13):
        sl = slice(hh * d, (hh + 1) * d)
        assert normwise_err(got[:, sl], want[:, sl]) <= FLUX_ATTN_TOL, hh


def form(t, h):
    """(waves of a workgroup, blocks cut between two of them) on this device."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    small, large = h * -(-t // 128), h * -(-t // 256)
    if t <= 128 or small <= cus or (small <= 2 * cus and large > cus):
        return 4, False
    return 8, large > cus


# Values in the first, second, a middle and the last tile of 32 keys, in 4-wave
# blocks and 8-wave ones, whole and cut between two workgroups.
FORMS = [(300, 4, 128, 4, False), (300, 4, 40, 4, False), (512, 100, 128, 8, False), (700, 100, 128, 8, True),
         (700, 100, 64, 8, True), (1200, 60, 32, 8, True)]


@pytest.mark.parametrize("t,h,d,waves,cut", FORMS)
@pytest.mark.parametrize("where", ["first", "second", "middle", "last"])
def test_flux_attention_wide_values_every_form(rt, t, h, d, waves, cut, where):
    if form(t, h) != (waves, cut):
        pytest.skip(f"{h} heads of {t} queries run as {form(t, h)} on this device")
    row = {"first": 0, "second": 40, "middle": t // 2, "last": t - 1}[where]
    test_flux_attention_values_without_limbs(rt, t, h, d, row)


def test_flux_attention_wide_values_cost(rt):
    """One infinity costs a call at most what f32 matrix steps do: 16 / 6 of the
    limbs' matrix time, less than 3 times the call, where loads from memory in
    place of the staged tiles took 5 to 9 times."""
    import torch
    t, h, d = 1280, 24, 128
    say(f"[flux wide cost] t={t} heads={h}")
    q, k, v = (to_dev(a) for a in rand(t, h, d))
    out = torch.empty_like(q)

    def time_of():
        best = 1e9
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                rt.flux_attention(q, k, v, h, d, out=out)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    clean = time_of()
    v[0, ::d] = float("inf")  # every head's first value: every block is in f32 throughout
    assert time_of() <= 3.5 * clean


@pytest.mark.parametrize("t,h,d,row", [(300, 4, 128, 0), (300, 4, 128, 290), (300, 4, 40, 64), (800, 70, 128, 31),
                                       (800, 70, 128, 799), (700, 100, 64, 350)])
def test_flux_attention_values_without_limbs(rt, t, h, d, row):
    say(f"[flux limbs wide] t={t} heads={h} head_dim={d} row={row}")
    q, k, v = rand(t, h, d)
    head = [slice(i * d, (i + 1) * d) for i in range(4)]
    # head 0: an infinity and a NaN in v reach their columns of every row
    v[row, 3], v[row, 5] = np.inf, np.nan
    # head 1: products that overflow downwards drop the key, here in every row
    q[:, head[1]] = 0.0
    q[:, head[1].start + 1] = np.float32(1.7e25)
    k[:, head[1].start + 1] = 0.0
    k[row, head[1].start + 1] = np.float32(-1.3e19)
    # head 2: a key that meets tiny queries with huge values
    q[:, head[2].start] = np.float32(1e-38)
    k[row, head[2].start] = np.float32(3.4e38)
    # head 3: an infinite v, one of opposite sign next to it, and one huge query
    v[row, head[3].start] = -np.inf
    q[0, head[3]] = 0.0
    q[0, head[3].start + 1] = np.float32(3e37)
    k[:, head[3].start + 1] = np.where(np.arange(t) == row, 1e-37, -1e-37)
    got, want = run(rt, q, k, v, h, d), exact(q, k, v, h, d)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.isposinf(got), np.isposinf(want))
        assert np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    for sl in head + [slice(4 * d, h * d)]:
        if sl.stop > sl.start:
            g, w, f = got[:, sl], want[:, sl], fin[:, sl]
            assert normwise_err(np.where(f, g, 0), np.where(f, w, 0)) <= FLUX_ATTN_TOL


@pytest.mark.parametrize("scale", [1e-30, 1e18])
def test_flux_attention_scaled_values(rt, scale):
    t, h, d = 300, 4, 64
    say(f"[flux limbs scaled] v x {scale}")
    q, k, v = rand(t, h, d)
    v = (v * np.float32(scale)).astype(np.float32)
    assert normwise_err(run(rt, q, k, v, h, d), exact(q, k, v, h, d)) <= FLUX_ATTN_TOL


# (2^100: normwise_err measures against 1e-30 at least)
@pytest.mark.parametrize("t,h,d", [(300, 4, 64), (700, 100, 128), (512, 100, 32)])
@pytest.mark.parametrize("scale", [1e-33, 1e-35, 1e-37])
def test_flux_attention_tiny_columns(rt, t, h, d, scale):
    """v of f32's smallest normal values in some dims keeps f32's bits there,
    beside ordinary dims."""
    say(f"[flux limbs tiny] t={t} heads={h} head_dim={d} v x {scale}")
    q, k, v = rand(t, h, d)
    tiny = np.arange(h * d) % 3 == 0
    v = np.where(tiny, v * np.float32(scale), v).astype(np.float32)
    got, want = run(rt, q, k, v, h, d), exact(q, k, v, h, d)
    assert normwise_err(got[:, ~tiny], want[:, ~tiny]) <= FLUX_ATTN_TOL
    assert normwise_err(got[:, tiny] * 2.0 ** 100, want[:, tiny] * 2.0 ** 100) <= FLUX_ATTN_TOL


def test_flux_attention_tiny_weights(rt):
    """Weights of 2^-122 on every key that has a value keep f32's bits.  Bound: a
    weight's exponent of 122 rounds by 122 * 2^-24 = 7.3e-6 in q and as much in
    the subtracted maximum."""
    t, h, d = 600, 3, 64
    say("[flux limbs tiny] weights")
    q, k, v = rand(t, h, d)
    q[:], k[:] = 0.0, 0.0
    q[:, ::d], k[:, ::d] = 8.0, -42.25
    k[77, ::d], v[77] = 42.25, 0.0
    got, want = run(rt, q, k, v, h, d), exact(q, k, v, h, d)
    assert 0 < np.abs(want).max() < 1e-33
    assert normwise_err(got * 2.0 ** 120, want * 2.0 ** 120) <= 2e-5


def test_flux_attention_captured_without_workspace(rt):
    say("[flux limbs] captured without workspace")
    run_case("flux")
