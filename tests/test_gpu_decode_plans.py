"""Decode rows at the edges of their launch plan: caches past 256 MB
(non-temporal K/V loads) with a last tile that is not full, at a capacity the
device key count stays below, more row tiles than resident workgroups, one key;
against float64 attention (tolerance: the layer's parity bar)."""

import pytest
import torch

from helpers import assert_close, np64

pytestmark = pytest.mark.gpu


def _case(B, H, Hkv, n, cap, D, dtype, dev_count, add=False):
    from delta_attention import ops
    g = torch.Generator(device="cuda").manual_seed(n + D)
    q = torch.randn(B, 1, H, D, device="cuda", generator=g).to(dtype).transpose(1, 2)
    k = torch.randn(B, cap, Hkv, D, device="cuda", generator=g, dtype=dtype).transpose(1, 2)
    v = torch.randn(B, cap, Hkv, D, device="cuda", generator=g, dtype=dtype).transpose(1, 2)
    scale = D ** -0.5
    if dev_count:
        nk = torch.full((1,), n, dtype=torch.int32, device="cuda")
        extra = torch.randn(B, H, 1, D, device="cuda", generator=g).to(dtype) if add else None
        out = ops.decode_attention(q, k, v, window=0, sink=0, sm_scale=scale, n_keys=nk, add=extra)
    else:
        out = ops.decode_attention(q, k[:, :, :n], v[:, :, :n], window=0, sink=0, sm_scale=scale)
    G = H // Hkv
    ref = torch.empty(B, H, 1, D, dtype=torch.float64)
    for b in range(B):
        for h in range(Hkv):
            kk, vv = k[b, h, :n].double().contiguous(), v[b, h, :n].double().contiguous()
            s = kk @ q[b, h * G:(h + 1) * G, 0].double().t().contiguous() * scale
            ref[b, h * G:(h + 1) * G, 0] = (torch.softmax(s, 0).t().contiguous() @ vv).cpu()
    if add:
        ref = ref + extra.double().cpu()
    assert_close(np64(out), ref.numpy(), what=f"decode B{B} H{H}/{Hkv} n{n} D{D} {dtype}")


@pytest.mark.parametrize("B,H,Hkv,n,cap,D,dtype,dev_count", [
    (1, 16, 8, 66001, 66001, 128, torch.bfloat16, False),
    (1, 16, 8, 40, 66001, 128, torch.float16, True),      # far fewer keys than the capacity
    (2, 8, 4, 33100, 33200, 256, torch.bfloat16, False),
    (3, 10, 2, 90011, 90011, 128, torch.float16, False),  # five heads per kv head
    (1, 32, 16, 70000, 70000, 64, torch.bfloat16, False),
    (70, 8, 8, 100, 100, 32, torch.bfloat16, False),      # 560 row tiles: no split
    (9, 8, 8, 2700, 2700, 64, torch.bfloat16, False),     # several splits, one round
    (1, 2, 1, 1, 1, 64, torch.bfloat16, False),
])
def test_decode_plan_edges(gpu, B, H, Hkv, n, cap, D, dtype, dev_count):
    _case(B, H, Hkv, n, cap, D, dtype, dev_count)


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("B,H,Hkv,n,dtype,add", [
    (1, 8, 8, 700, torch.bfloat16, True),          # 16 threads a task, few tasks
    (2, 32, 8, 5000, torch.float16, True),         # at head_dim 128 the most threads of the 4-column merge
    (3, 32, 8, 5000, torch.bfloat16, False),       # past them
    (4, 20, 4, 100, torch.float16, True),          # two splits
])
def test_merge_widths(gpu, B, H, Hkv, n, D, dtype, add):
    """Both merge kernels over float partials (4 and 8 columns a task), with the
    cached delta's add."""
    _case(B, H, Hkv, n, n + 60, D, dtype, True, add)
