"""Captures that find no workspace, each in a process of its own: the library's
workspace is per process and never shrinks, so inside a test run earlier tests
have grown it past any need.  Run as a script with a case's name; run_case()
starts it and checks that it got to its end."""
import os
import subprocess
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))


def run_case(name):
    out = subprocess.run([sys.executable, os.path.abspath(__file__), name], capture_output=True, text=True, timeout=100,
                         cwd=HERE)
    assert out.returncode == 0 and f"{name}: done" in out.stdout, out.stdout + out.stderr


def replays(rt, fn, out, check):
    """fn captured with the workspace as it is; check(out) after each of three replays."""
    import torch
    torch.cuda.synchronize()
    before = rt.workspace_bytes()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    assert rt.workspace_bytes() == before
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        check(out)


def gemv_q4_0(rt):
    import torch
    from helpers import GEMV_TOL, from_dev, normwise_err, to_dev
    n, k, m = 64, 12288, 8
    rng = np.random.default_rng(5)
    b = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
    b[:, :2] = (0.002 + 0.004 * rng.random(b.shape[0])).astype(np.float16)[:, None].view(np.uint8)
    q = np.concatenate([b[:, 2:] & 15, b[:, 2:] >> 4], 1).astype(np.float64) - 8
    v = (q * b[:, :2].copy().view(np.float16).astype(np.float64)).reshape(n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w, dx, y = to_dev(b.reshape(-1)), to_dev(x), torch.zeros((m, n), device="cuda")
    rt.gemv(rt.Q4_0, w, dx[:, :256].contiguous(), n, 256)  # (loads the kernels; K of one slot takes no scratch)
    assert rt.library().lib.rt_hip_gemv_workspace_bytes(rt.Q4_0, n, k, m) > rt.workspace_bytes()

    def check(y):
        assert normwise_err(from_dev(y), x.astype(np.float64) @ v.T) <= GEMV_TOL

    replays(rt, lambda: rt.gemv(rt.Q4_0, w, dx, n, k, y=y), y, check)


def gemm(rt, a_bf16):
    import torch
    from helpers import GEMM_TOL_SAME_OPERANDS, from_dev, normwise_err, same_operand_err
    m, n, k = 200, 256, 1152
    g = torch.Generator(device="cuda").manual_seed(2)
    a = torch.randn((m, k), device="cuda", generator=g)
    a = a.to(torch.bfloat16) if a_bf16 else a
    w = (torch.randn((n, k), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    c = torch.zeros((m, n), device="cuda")
    rt.gemm(rt.BF16, a[:9, :64].contiguous(), w[:, :64].contiguous().view(torch.int16), n, 64)
    need = rt.library().lib.rt_hip_gemm_workspace_bytes(rt.BF16, rt.BF16 if a_bf16 else rt.F32, m, n, k)
    assert need > rt.workspace_bytes()

    def check(c):
        assert same_operand_err(c, a, w) <= GEMM_TOL_SAME_OPERANDS

    replays(rt, lambda: rt.gemm(rt.BF16, a, w.view(torch.int16), n, k, c=c), c, check)
    eager = from_dev(rt.gemm(rt.BF16, a, w.view(torch.int16), n, k))
    assert rt.workspace_bytes() >= need and normwise_err(from_dev(c), eager) <= GEMM_TOL_SAME_OPERANDS


def gemm_4bit(rt, fmt):
    """Room for the widened weight alone."""
    import torch
    from helpers import GEMM_TOL_SAME_OPERANDS, same_operand_err
    m, n, k = 300, 1024, 1088
    rng = np.random.default_rng(k)
    if fmt == "q4mat":
        code = rt.Q4MAT
        w = rt.q4mat_upload(rng.integers(0, 256, n * k // 2, dtype=np.uint8),
                            (0.01 * rng.random(n * k // 32)).astype(np.float32), n, k)
    else:
        code = rt.Q4_0
        b = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
        b[:, :2] = np.float16(0.01).reshape(1).view(np.uint8)
        w = torch.from_numpy(b.reshape(-1)).cuda()
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    c = torch.zeros((m, n), device="cuda")
    wide = rt.dequant(code, w, n, k, bf16=True).view(torch.bfloat16)
    bits = wide[:, :64].contiguous().view(torch.int16)
    rt.gemm(rt.BF16, a[:9, :64].contiguous(), bits, n, 64)
    rt.reserve_workspace(n * k * 2)
    assert rt.library().lib.rt_hip_gemm_workspace_bytes(code, rt.F32, m, n, k) > rt.workspace_bytes() >= n * k * 2

    def check(c):
        assert same_operand_err(c, a, wide) <= GEMM_TOL_SAME_OPERANDS

    replays(rt, lambda: rt.gemm(code, a, w, n, k, c=c), c, check)


def flux(rt):
    import torch
    from helpers import from_dev, normwise_err, to_dev
    from test_gpu_flux_attention_limbs import FLUX_ATTN_TOL, exact, rand
    t, h, d = 700, 100, 128
    q, k, v = rand(t, h, d)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    out = torch.zeros_like(dq)
    rt.flux_attention(dq[:64, :d].contiguous(), dk[:64, :d].contiguous(), dv[:64, :d].contiguous(), 1, d)
    assert rt.library().lib.rt_hip_flux_attention_workspace_bytes(t, h, d) > rt.workspace_bytes()
    want = exact(q, k, v, h, d)

    def check(out):
        assert normwise_err(from_dev(out), want) <= FLUX_ATTN_TOL

    replays(rt, lambda: rt.flux_attention(dq, dk, dv, h, d, out=out), out, check)


def failed_growth(rt):
    """A workspace that cannot be allocated is an error of that call alone."""
    import torch
    y = rt.gemv(rt.BF16, torch.zeros((16, 256), dtype=torch.int16, device="cuda"), torch.ones((2, 256), device="cuda"),
                16, 256)
    try:
        rt.reserve_workspace(1 << 46)
        raise AssertionError("64 TiB of workspace")
    except rt.RtHipError as e:
        assert e.code == 4  # RT_HIP_E_OOM
    x = torch.ones((2, 256), device="cuda")
    rt.gemv(rt.BF16, torch.zeros((16, 256), dtype=torch.int16, device="cuda"), x, 16, 256, y=y)
    assert (y == 0).all()


CASES = {"gemv_q4_0": gemv_q4_0, "gemm_f32": lambda rt: gemm(rt, False), "gemm_bf16": lambda rt: gemm(rt, True),
         "gemm_q4_0": lambda rt: gemm_4bit(rt, "q4_0"), "gemm_q4mat": lambda rt: gemm_4bit(rt, "q4mat"), "flux": flux,
         "failed_growth": failed_growth}

if __name__ == "__main__":
    sys.path.insert(0, HERE)
    import torch
    assert torch.cuda.is_available()  # (torch's HIP runtime first: the library joins it)
    from conftest import load_package
    package = load_package().rt_hip
    package.init(0)
    CASES[sys.argv[1]](package)
    print(f"{sys.argv[1]}: done", flush=True)
