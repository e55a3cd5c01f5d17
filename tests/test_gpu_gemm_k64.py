"""BF16 GEMM with K % 64 == 0 but not % 256: the pipelined kernels at step
counts of every remainder mod 4, with and without K splits, on 128- and
256-row tiles; the Q4_0 / Q4Mat weights that are widened first; and a capture
that finds no workspace, which takes the kernel that needs none.

Bound: GEMM_TOL_SAME_OPERANDS, the f32 accumulation of the same bf16-rounded
operands against float64 (as test_gpu_gemm.py)."""
import numpy as np
import pytest

from fresh_process import run_case
from helpers import GEMM_TOL_SAME_OPERANDS, same_operand_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,a_bf16", [(9, 64, 64, False), (128, 132, 192, True), (129, 1152, 1152, False),
                                          (333, 256, 320, True), (700, 1024, 1088, False), (60, 3072, 2880, False),
                                          (4100, 4000, 448, True), (4097, 4100, 1152, False)])
def test_bf16_gemm_k64(rt, m, n, k, a_bf16):
    import torch
    say(f"[gemm k64] {m} x {n} x {k} a_bf16={a_bf16}")
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn((m, k), device="cuda", generator=g)
    if a_bf16:
        a = a.to(torch.bfloat16)
    w = (torch.randn((n, k), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    bias = torch.randn((n,), device="cuda", generator=g)
    c = rt.gemm(rt.BF16, a, w.view(torch.int16), n, k, bias=bias)
    assert same_operand_err(c - bias, a, w) <= 2 * GEMM_TOL_SAME_OPERANDS  # 2: the bias subtracted again in f32


# Few rows and at most three steps of K take the kernel without a pipeline:
# both sides of each line, and the one-slice launches of short K.
@pytest.mark.parametrize("m,n,k,a_bf16", [(9, 68, 64, False), (48, 132, 128, False), (49, 132, 128, False),
                                          (9, 132, 192, True), (32, 1024, 192, True), (33, 1024, 192, True),
                                          (9, 1024, 192, False), (300, 1028, 128, True), (1000, 516, 128, False)])
def test_bf16_gemm_short_k(rt, m, n, k, a_bf16):
    test_bf16_gemm_k64(rt, m, n, k, a_bf16)


def test_bf16_gemm_short_k_cost(rt):
    """K of two steps over many rows is not summed from slices of one step: it
    costs less than K of eight."""
    import torch
    say("[gemm k64] short K cost")
    m = n = 1024

    def time_of(k):
        a = torch.randn((m, k), device="cuda").bfloat16()
        w = torch.randn((n, k), device="cuda").bfloat16()
        c, best = torch.empty((m, n), device="cuda"), 1e9
        for _ in range(6):
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            for _ in range(50):
                rt.gemm(rt.BF16, a, w.view(torch.int16), n, k, c=c)
            e.record()
            torch.cuda.synchronize()
            best = min(best, s.elapsed_time(e))
        return best

    assert rt.library().lib.rt_hip_gemm_workspace_bytes(rt.BF16, rt.BF16, m, n, 128) == 0
    assert time_of(128) < time_of(512)


@pytest.mark.parametrize("fmt,k", [("q4_0", 320), ("q4mat", 1152)])
def test_4bit_gemm_k64(rt, fmt, k):
    import torch
    m, n = 300, 260
    say(f"[gemm k64 {fmt}] {m} x {n} x {k}")
    rng = np.random.default_rng(k)
    if fmt == "q4mat":
        code = rt.Q4MAT
        w = rt.q4mat_upload(rng.integers(0, 256, n * k // 2, dtype=np.uint8),
                            (0.01 * rng.random(n * k // 32)).astype(np.float32), n, k)
    else:
        code = rt.Q4_0
        b = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
        b[:, :2] = np.float16(0.01) .reshape(1).view(np.uint8)
        w = torch.from_numpy(b.reshape(-1)).cuda()
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    wide = rt.dequant(code, w, n, k, bf16=True).view(torch.bfloat16)
    assert same_operand_err(rt.gemm(code, a, w, n, k), a, wide) <= GEMM_TOL_SAME_OPERANDS


@pytest.mark.parametrize("case", ["gemm_f32", "gemm_bf16", "gemm_q4_0", "gemm_q4mat"])
def test_gemm_k64_captured_without_workspace(rt, case):
    say(f"[gemm k64] captured without workspace: {case}")
    run_case(case)
