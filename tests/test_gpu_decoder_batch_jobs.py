"""The decoder's batched step where several projections share a launch and a
residual add shares one with the next norm: 2 to 8 rows, q/k/v widths whose
boundaries fall inside a workgroup's tiles, BF16 layers that leave one or no
Q4_K projection to share, and each hidden width class of the norm kernel.

Bound: STEP_TOL of test_gpu_decoder.py against the oracle's single steps."""
import numpy as np
import pytest

from helpers import normwise_err, say
from test_gpu_decoder import GEMMA, LLAMA, STEP_TOL, Model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arch,rows,wide,cfg", [
    ("llama", 8, None, dict(n_heads=4, n_kv_heads=1)),
    ("llama", 2, set(), dict(hidden=4608, n_heads=4, n_kv_heads=2, ffn=512)),
    ("llama", 3, {0, 1}, dict(hidden=1024)),
    ("gemma3", 5, {1}, dict(hidden=6144, n_heads=2, n_kv_heads=1, ffn=256)),
    ("llama", 6, set(), dict(hidden=8448, n_heads=4, n_kv_heads=2, ffn=256)),
    ("gemma3", 7, set(), dict(hidden=2560, ffn=2048, n_heads=4, n_kv_heads=2)),
])
def test_decoder_batch_shared_launches(rt, orc, arch, rows, wide, cfg):
    cfg = dict(GEMMA if arch == "gemma3" else LLAMA, max_batch=rows, vocab=200, **cfg)
    say(f"[decoder batch jobs] {arch} rows={rows} hidden={cfg['hidden']}")
    rng = np.random.default_rng(rows)
    m = Model(orc, arch, rng, wide_layers=wide, **cfg)
    dec = m.load(rt)
    try:
        tokens = rng.integers(0, cfg["vocab"], 2 * rows)
        want = [m.step(int(t), pos) for pos, t in enumerate(tokens)]
        for first in (0, rows):  # twice: the second replays the graph
            got = dec.step_batch(tokens[first:first + rows], first)
            for i in range(rows):
                assert normwise_err(got[i], want[first + i]) <= STEP_TOL, (first, i)
    finally:
        dec.close()
