"""Backward launches at the edges of their item plans: short row lists beside
long ones (dq splits past the end of a list), key blocks cut into 96-row
chunks with a remainder, one tile, and launches just past one round of
workgroups; gradients against float64 autograd of masked softmax attention.
Bound: P and dS enter the products in 16 bits, gradients are sums of such
products rounded once: the bar of test_gpu_train.py."""

import pytest
import torch

from helpers import np64

pytestmark = pytest.mark.gpu


def _ref(q, k, v, up, vis, scale):
    q, k, v = (t.double().cpu().requires_grad_(True) for t in (q, k, v))
    G = q.shape[1] // k.shape[1]
    kk, vv = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    s = (q @ kk.transpose(2, 3)) * scale
    p = torch.softmax(s.masked_fill(~vis.cpu(), float("-inf")), -1)
    out = (p @ vv).transpose(1, 2)
    return torch.autograd.grad(out, (q, k, v), up.double().cpu())


def _close(got, ref, what):
    for g, r, n in zip(got, ref, ("dq", "dk", "dv")):
        a, b = np64(g).ravel(), r.numpy().ravel()
        cos = float(a @ b / ((a @ a) ** 0.5 * (b @ b) ** 0.5))
        err, bound = float(abs(a - b).max()), 2e-2 * max(1.0, float(abs(b).max()))
        print(f"{what} {n}: cos {cos:.6f} max|err| {err:.4g}", flush=True)
        assert cos >= 0.999 and err <= bound, (what, n, cos, err, bound)


def _inputs(B, H, Hkv, S, D, dtype, n):
    g = torch.Generator().manual_seed(S + D)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    return r(B, H, S, D), r(B, Hkv, S, D), r(B, Hkv, S, D), r(B, n, H, D)


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype,rows", [
    (1, 8, 2, 2100, 64, torch.bfloat16, list(range(0, 700, 9)) + list(range(2000, 2100))),
    (2, 4, 4, 1000, 128, torch.float16, list(range(0, 900, 16)) + list(range(900, 1000))),
    (1, 4, 2, 64, 32, torch.bfloat16, list(range(64))),          # one tile
    (1, 5, 1, 900, 128, torch.bfloat16, [0, 1, 63, 64, 255, 256, 257, 899]),
    (1, 8, 8, 1300, 64, torch.bfloat16, list(range(0, 1300, 3))),
    (1, 5, 1, 1300, 128, torch.bfloat16, list(range(300, 1300, 3))),     # first keys seen by every row
    (2, 8, 1, 700, 128, torch.float16, list(range(0, 700, 64)) + list(range(690, 700))),
    (1, 2, 2, 300, 128, torch.bfloat16, list(range(300))),               # every row
    (1, 3, 3, 500, 128, torch.bfloat16, [499]),
])
def test_rows(gpu, B, H, Hkv, S, D, dtype, rows):
    from delta_attention import ops
    idx = torch.tensor(rows, device="cuda")
    q, k, v, up = _inputs(B, H, Hkv, S, D, dtype, len(rows))
    scale = D ** -0.5
    out, lse = ops.rows_attention_lse(q, k, v, idx, scale)
    got = ops.rows_attention_bwd(q, k, v, idx, out, up, lse, sm_scale=scale)
    vis = torch.arange(S, device="cuda")[None] <= idx[:, None]
    rq, rk, rv = _ref(q[:, :, idx], k, v, up, vis, scale)
    _close((got[0][:, :, idx], got[1], got[2]), (rq, rk, rv), f"rows S{S} D{D} n{len(rows)}")


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype,window,sink", [
    (1, 4, 1, 1000, 64, torch.bfloat16, 200, 70),      # 96-row chunks, last one short
    (1, 2, 2, 400, 128, torch.float16, 1000, 0),       # window past the sequence
    (2, 8, 2, 640, 32, torch.bfloat16, 128, 300),      # three sink blocks
    (1, 4, 4, 96, 64, torch.bfloat16, 64, 8),          # one key block
    # head_dim 128 (the unit ring of dkdv_pipe_kernel): five heads and a last
    # step of 8 rows, eight heads, one head with fewer units than ring slots,
    # a window shorter than its block, sinks ending inside a wave's keys
    (1, 5, 1, 1000, 128, torch.bfloat16, 300, 70),
    (2, 8, 1, 500, 128, torch.float16, 128, 0),
    (1, 3, 3, 70, 128, torch.bfloat16, 64, 0),
    (1, 2, 1, 333, 128, torch.bfloat16, 40, 45),
    (1, 4, 2, 2100, 128, torch.bfloat16, 256, 128),
])
def test_key_sparse(gpu, B, H, Hkv, S, D, dtype, window, sink):
    from delta_attention import ops
    q, k, v, up = _inputs(B, H, Hkv, S, D, dtype, S)
    scale = D ** -0.5
    out, lse = ops.sparse_attention_lse(q, k, v, window=window, sink=sink, sm_scale=scale)
    got = ops.sparse_attention_bwd(q, k, v, out, up, lse, window=window, sink=sink, sm_scale=scale)
    r = torch.arange(S, device="cuda")
    lo = r // 64 * 64 + 64 - window
    vis = (r[None] <= r[:, None]) & ((r[None] < sink) | (r[None] >= lo[:, None]))
    _close(got, _ref(q, k, v, up, vis, scale), f"key-sparse S{S} D{D}")
