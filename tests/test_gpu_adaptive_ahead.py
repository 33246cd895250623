"""The adaptive layer's rows ahead when the stride falls at once and comes back
to its start late."""

import pytest
import torch

from helpers import gen_qkv
from test_gpu_layer import _cfg

pytestmark = pytest.mark.gpu


def test_late_stride_takes_rows_ahead(gpu):
    """Scores of four times the variance in chunks 0 - 4 (their deltas point
    everywhere: the stride falls from 32 to 8), flat ones and sink values far
    from the others' from chunk 5 on (deltas alike: it doubles per chunk). From
    chunk 8 on the anchors' dense rows come from one launch, with the splits of
    a launch over every multiple of 32 (33 key tiles) and not those of a chunk's
    own (4 tiles): the layer's output has the bits of the composition from such
    a launch (fp16, whose rounding shows the two launches' fp32 merges apart)."""
    from delta_attention import ops
    from delta_attention.llama import LlamaAttention
    H, Hkv, D, s, chunk, gamma0, gmin, window, sink = 32, 8, 128, 10500, 512, 32, 8, 256, 16
    late, first, dtype = 5, 8, torch.float16
    scale = D ** -0.5
    q, k, v = gen_qkv(1, H, Hkv, s, D, seed=41, dtype=torch.float32)
    q[:, :, :late * chunk] *= 4.0
    q[:, :, late * chunk:] *= 0.05
    v[:, :, :sink] += 8.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    cfg = _cfg(H, Hkv, D, stride_policy="adaptive", adapt_chunk=chunk, delta_lambda=gamma0,
               gamma_min=gmin, gamma_max=128, sliding_window=window, sink_tokens=sink)
    m = LlamaAttention(cfg, layer_idx=0).cuda().to(dtype)
    out, _ = m.delta_forward(m, q, k, v, None, scaling=scale)
    chunks = m._stride_stats["chunks"]
    gammas = [c["gamma"] for c in chunks]
    print("strides", gammas, flush=True)
    assert min(gammas) == gmin and all(g >= gamma0 for g in gammas[first:]) and gammas[first - 2] < gamma0
    s_p = s - (s % gamma0 + 128)
    sparse = ops.sparse_attention(q, k, v, window=window, sink=sink, sm_scale=scale)
    rows = torch.arange(0, s_p, gamma0, device="cuda")
    ahead = ops.qsparse_attention(q, k[:, :, :s_p], v[:, :, :s_p], rows, scale, q_rows=rows)
    n_live, max_n = chunk // gamma0, chunk // gmin
    differ = False
    for ci, c in enumerate(chunks):
        start, g, n = c["start"], c["gamma"], c["n_anchors"]
        end = min(start + chunk, s_p)
        anchors = torch.arange(start, end, g, device="cuda")
        padded = torch.full((max_n,), -1, dtype=torch.int64, device="cuda")
        padded[:n] = anchors
        own = ops.qsparse_attention(q, k[:, :, :end], v[:, :, :end], padded, scale, q_rows=padded,
                                    n_live=n_live,
                                    n_dev=torch.tensor([n], dtype=torch.int32, device="cuda"))[:, :, :n]
        dense = own
        if ci >= first:
            dense = ahead[:, :, start // gamma0::g // gamma0][:, :, :n]
            differ = differ or not torch.equal(dense, own)
        delta = dense.transpose(1, 2) - sparse[:, anchors]
        owner = torch.div(torch.arange(end - start, device="cuda"), g, rounding_mode="floor")
        assert torch.equal(out[:, start:end], sparse[:, start:end] + delta[:, owner]), (ci, g)
    assert differ      # the two launches round some rows differently
