"""head_dim 256 at the edges of its tile loop: one to five 64-key tiles with
and without a remainder, single rows and row counts around a 128-row tile, and
inputs whose reference maxima move, against the oracle's softmax (tolerance: the layer's parity bar, helpers.assert_close)."""

import numpy as np
import pytest
import torch

from helpers import assert_close, gen_qkv, np64
from oracle import delta_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,N", [(1, 1), (1, 64), (3, 65), (31, 128), (33, 129), (64, 192), (65, 257),
                                 (129, 320)])
def test_rows(gpu, n, N, dtype):
    from delta_attention.delta_kernel import attention
    q, k, v = gen_qkv(2, 4, 2, N, 256, seed=N, dtype=dtype, model_layout=True)
    rows = torch.arange(N - n, N, device="cuda")
    out = attention(q[:, :, rows], k, v, rows[None], 256 ** -0.5)
    ref = O.qsparse_attention(np64(q)[:, :, N - n:], np64(k), np64(v), rows.cpu().numpy(), 256 ** -0.5)
    assert_close(np64(out), ref, what=f"rows d256 n{n} N{N} {dtype}")


@pytest.mark.parametrize("kind", ["growing", "outliers"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_exact_pass(gpu, kind, dtype):
    """Key norms growing 12x along the sequence, or 1 % of the keys at 40x:
    every row keeps the same bits whichever rows share its workgroup, also where
    their reference maxima move."""
    from delta_attention import ops
    from delta_attention.delta_kernel import attention
    from delta_attention.llama import repeat_kv
    S, scale = 900, 256 ** -0.5
    q, k, v = gen_qkv(1, 4, 2, S, 256, seed=5, dtype=torch.float32)
    if kind == "growing":
        k = k * torch.linspace(1.0, 12.0, S, device="cuda")[None, None, :, None]
    else:
        k[:, :, torch.randperm(S, generator=torch.Generator().manual_seed(6))[:9].cuda()] *= 40.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    rows = np.arange(0, S, 7)
    rt = torch.from_numpy(rows)[None].cuda()
    got = attention(q[:, :, rows], k, v, rt, scale)
    assert torch.equal(got, attention(q[:, :, rows], repeat_kv(k, 2), repeat_kv(v, 2), rt, scale))
    assert_close(np64(got), O.qsparse_attention(np64(q)[:, :, rows], np64(k), np64(v), rows, scale),
                 what=f"rows d256 {kind} {dtype}")
    sp = ops.sparse_attention(q, k, v, window=256, sink=16, sm_scale=scale)
    assert_close(np64(sp), O.sparse_attention(np64(q), np64(k), np64(v), 256, 16, scale),
                 what=f"key-sparse d256 {kind} {dtype}")


def test_moving_maxima_cost_no_second_pass(gpu):
    """Keys whose norms grow 12x along the sequence move every row's reference
    max. The key-sparse launch still computes its tiles once: at most 1.5 times
    as long as on keys of one norm (two passes: 2.05 times; the smallest of
    several batches of launches each)."""
    from delta_attention import ops
    S, scale = 8009, 256 ** -0.5
    q, k, v = gen_qkv(1, 16, 4, S, 256, seed=7)
    grow = (k.float() * torch.linspace(1.0, 12.0, S, device="cuda")[None, None, :, None]).to(k.dtype)

    def us(kk):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = float("inf")
        for _ in range(6):
            a.record()
            for _ in range(20):
                ops.sparse_attention(q, kk, v, window=2048, sink=128, sm_scale=scale)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 50)
        return best

    flat, moving = us(k), us(grow)
    print(f"d256 key-sparse: one norm {flat:.1f} us, growing {moving:.1f} us", flush=True)
    assert moving <= 1.5 * flat, (flat, moving)
