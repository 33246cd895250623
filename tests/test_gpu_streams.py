"""Launches follow torch's current stream: the raw stream handle the bindings
pass, and the row lists kept per size and stream by the training path."""

import pytest
import torch

from helpers import gen_qkv

pytestmark = pytest.mark.gpu


def test_side_stream_matches_default(gpu):
    from delta_attention import ops
    from delta_attention.train.flex_delta import delta_forward_train
    q, k, v = gen_qkv(1, 4, 2, 512, 64, seed=9)
    ts = [t.requires_grad_(True) for t in (q, k, v)]

    def step():
        out = delta_forward_train(*ts, 16, 128, 16)
        dec = ops.decode_attention(q.detach()[:, :, -1:], k.detach(), v.detach(), window=128, sink=16,
                                   sm_scale=0.125)
        return (out.detach(), dec, *torch.autograd.grad(out, ts, torch.ones_like(out)))

    ref = step()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    assert ops._stream(q.device) == torch.cuda.current_stream().cuda_stream
    here = ops.selected_rows_here(512, 16, q.device)
    with torch.cuda.stream(side):
        assert ops._stream(q.device) == side.cuda_stream
        there = ops.selected_rows_here(512, 16, q.device)
        got = step()
    side.synchronize()
    assert here is ops.selected_rows_here(512, 16, q.device)
    assert there.data_ptr() != here.data_ptr() and torch.equal(there, here)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
