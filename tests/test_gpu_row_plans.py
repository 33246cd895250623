"""Selected-rows launches at the edges of their split plan: lists of one tile,
lists cut into the shortest items, a plan of exactly one item per resident
workgroup, one item per row tile, and the longest items of rows that end the
sequence; against the oracle (tolerance: the layer's parity bar)."""

import numpy as np
import pytest
import torch

from helpers import assert_close, gen_qkv, np64
from oracle import delta_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,n,N,D", [
    (1, 2, 2, 5, 40, 64),         # one key tile
    (1, 8, 2, 17, 600, 64),       # the shortest items: two of ten tiles
    (1, 8, 2, 33, 8000, 128),     # seven-tile items of 125
    (1, 8, 8, 1000, 1100, 128),   # 64 row tiles, eight splits: every slot one item
    (1, 8, 8, 1000, 1100, 256),   # the same at one workgroup per CU: four splits
    (64, 8, 8, 2, 1200, 32),      # 512 row tiles: one item each
    (65, 8, 8, 2, 1200, 32),      # one row tile past the slots
    (64, 8, 8, 2, 5200, 32),      # rows that end the sequence, one 82-tile item each
])
@pytest.mark.parametrize("selected", [False, True])
def test_plan_edges(gpu, B, H, Hkv, n, N, D, selected):
    """The same rows as the last n rows of a sequence (no q_rows) and as rows
    selected from a full q; both plans against the oracle on two batches."""
    from delta_attention import ops
    q, k, v = gen_qkv(B, H, Hkv, n, D, seed=N + D, N=N)
    rows = torch.arange(N - n, N, device="cuda")
    if selected:
        full = torch.zeros(B, H, N, D, dtype=q.dtype, device="cuda")
        full[:, :, N - n:] = q
        out = ops.qsparse_attention(full, k, v, rows, D ** -0.5, q_rows=rows)
    else:
        out = ops.qsparse_attention(q, k, v, rows[None], D ** -0.5)
    for b in {0, B - 1}:
        ref = O.qsparse_attention(np64(q[b:b + 1]), np64(k[b:b + 1]), np64(v[b:b + 1]),
                                  rows.cpu().numpy(), D ** -0.5)
        assert_close(np64(out[b:b + 1]), ref, what=f"B{B} n{n} N{N} D{D} batch {b}")


@pytest.mark.parametrize("n,N", [
    (64, 24000),      # row tiles just half full: one item per CU (31 of 12-13 tiles)
    (63, 24000),      # less than half full: two (15-tile items)
    (64, 65536),      # 16 tiles at two items per CU: one item of 32 tiles
    (64, 65537),      # 17 tiles: two items
])
def test_ending_rows_per_cu(gpu, n, N):
    """Rows that end a sequence around the rule for one or two items per CU."""
    from delta_attention import ops
    q, k, v = gen_qkv(1, 8, 8, n, 128, seed=N + n, N=N)
    rows = torch.arange(N - n, N, device="cuda")
    out = ops.qsparse_attention(q, k, v, rows[None], 128 ** -0.5)
    ref = O.qsparse_attention(np64(q), np64(k), np64(v), rows.cpu().numpy(), 128 ** -0.5)
    assert_close(np64(out), ref, what=f"n{n} N{N}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("gap", [10.0, 13.0])
def test_dominant_first_key(gpu, dtype, gap):
    """Key 0 stands `gap` nats above the mean score of every other key (whose
    scores are N(0, 1)) and has a zero value, so the output is the other keys'
    probabilities alone. In fp16 only the split that holds key 0 may pack them
    as subnormals (spacing 2^-24): with the 4-tile items of this plan 256 of
    12000 keys, each off by 2^-24 / sqrt(12) rms, against probabilities of
    2^(-gap / ln 2) e (rms over N(0, 1) scores), i.e. 4.1e-4 of the output at 13
    nats and less than that at 10; beside the rounding of the other
    probabilities and of the output, 2.5e-4 (fp16) or 2e-3 (bf16). Bound: twice
    the root of the sum of the squares."""
    from delta_attention import ops
    H, Hkv, D, N, n = 8, 2, 128, 12000, 64
    q, k, v = gen_qkv(1, H, Hkv, N, D, seed=3, dtype=torch.float32)
    q[..., 0] = 4.0
    k[..., 0] = 0.0
    k[:, :, 0] = 0.0
    k[:, :, 0, 0] = gap * D ** 0.5 / 4.0
    v[:, :, 0] = 0.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    rows = torch.arange(N - n, N, device="cuda")
    out = ops.qsparse_attention(q, k, v, rows, D ** -0.5, q_rows=rows)
    ref = O.qsparse_attention(np64(q)[:, :, N - n:], np64(k), np64(v), rows.cpu().numpy(), D ** -0.5)
    err = np.linalg.norm(np64(out).ravel() - ref.ravel()) / np.linalg.norm(ref)
    base = 2.5e-4 if dtype == torch.float16 else 2e-3
    sub = 4.1e-4 if dtype == torch.float16 else 0.0
    print(f"dominant first key {dtype} gap {gap}: rel {err:.3g}", flush=True)
    assert err <= 2 * (base ** 2 + sub ** 2) ** 0.5, err
