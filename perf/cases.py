"""What is measured of the delta-attention framework: the calls its users make,
from the smallest to the largest, each through a public entry point.

  prefill    ops.delta_prefill, one attention layer's prefill (modes "delta"
             and "recompute"; head_dim 64 / 128 / 256; bf16 and fp16)
  adaptive   LlamaAttention.delta_forward with stride_policy "adaptive"
  rows       delta_kernel.attention, query rows against a longer key range
             (a prompt chunk behind a cache, or selected rows of a prompt)
  decode     ops.decode_attention, one query row against a KV cache (sinks and
             a window, or every key)
  train      train.flex_delta.delta_forward_train with its backward
  layer      LlamaDecoderLayer.forward, a whole decoder layer's prefill

Inputs are N(0, 1) in the storage the model stack uses: [B, S, H, D]
projection outputs and [B, max_len, Hkv, D] caches, passed as transposed
views. Scores then have unit variance at sm_scale = D^-0.5.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "delta-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from delta_attention import ops  # noqa: E402
from delta_attention.delta_kernel import attention as rows_attention  # noqa: E402
from delta_attention.llama import LlamaAttention, rope_cos_sin  # noqa: E402
from delta_attention.model import LlamaConfig, LlamaDecoderLayer, init_weights_  # noqa: E402
from delta_attention.train.flex_delta import delta_forward_train  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
Q_BLOCK = 64      # the window is anchored at 64-row query blocks
ADAPT_CHUNK = 4096
GAMMA_MIN, GAMMA_MAX = 16, 256


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the smallest prompt with anchors: a short odd-length one on a small
        # head_dim-64 model, where launches and latency count
        dict(name="prefill_short_d64", kind="prefill", dtype="bf16", B=1, H=8, Hkv=2, D=64,
             S=1531, gamma=16, window=512, sink=64, mode="delta"),
        # a ragged batch-2 prompt, five query heads per kv head, wide window
        dict(name="prefill_ragged_gqa5", kind="prefill", dtype="bf16", B=2, H=40, Hkv=8, D=128,
             S=20011, gamma=64, window=4096, sink=64, mode="delta"),
        # a long-document layer, the headline geometry
        dict(name="prefill_128k", kind="prefill", dtype="bf16", B=1, H=32, Hkv=8, D=128,
             S=131072, gamma=64, window=2048, sink=128, mode="delta"),
        # mode "recompute" in fp16 with the reference's 1024 sinks and a stride
        # that is no power of two, odd length
        dict(name="prefill_recompute_fp16", kind="prefill", dtype="fp16", B=1, H=32, Hkv=8, D=128,
             S=28003, gamma=48, window=2048, sink=1024, mode="recompute"),
        # the adaptive stride, a ragged 40K prompt
        dict(name="adaptive_40k", kind="adaptive", dtype="bf16", B=1, H=32, Hkv=8, D=128,
             S=40009, gamma=64, window=2048, sink=128),
        # a follow-up prompt chunk behind a 16K cache, head_dim 256
        dict(name="rows_chunk_d256", kind="rows", dtype="bf16", B=1, H=16, Hkv=4, D=256,
             n=509, S=16901),
        # the sparse decode row: one token against sinks + window of a 32K
        # cache, the smallest call of all
        dict(name="decode_window", kind="decode", dtype="bf16", B=1, H=32, Hkv=8, D=128,
             S=32771, window=2048, sink=128),
        # the dense (anchor) decode row at a 128K context
        dict(name="decode_dense_128k", kind="decode", dtype="bf16", B=1, H=32, Hkv=8, D=128,
             S=131072, window=0, sink=0),
        # a batch of sequences decoding together, fp16, five heads per kv head
        dict(name="decode_batch_fp16", kind="decode", dtype="fp16", B=16, H=40, Hkv=8, D=128,
             S=6007, window=0, sink=0),
        # a training step's attention, forward and backward, long sequence
        dict(name="train_32k", kind="train", dtype="bf16", B=1, H=32, Hkv=8, D=128,
             S=32768, gamma=64, window=2048, sink=128),
        # the same on a small fp16 head_dim-64 model, batch 2, short sequences
        dict(name="train_short_d64_fp16", kind="train", dtype="fp16", B=2, H=8, Hkv=2, D=64,
             S=2048, gamma=16, window=512, sink=64),
        # a whole decoder layer (norms, projections, RoPE, delta attention,
        # MLP) over an ordinary odd-length prompt
        dict(name="layer_6k", kind="layer", dtype="bf16", B=1, H=32, Hkv=8, D=128,
             S=6001, gamma=64, window=2048, sink=128, hidden=4096, inter=14336),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: head geometries of the model
    configurations (GQA 1 to 8), lengths spread over their logarithm and
    mostly odd, every mode, stride, window and sink setting in use. It does
    at most half the largest listed case's work, train a sixth, head_dims
    other than 128 a fifth (their rates are lower)."""
    limit = work(next(c for c in listed() if c["name"] == "prefill_128k"))
    while True:
        c = _draw_once(rng)
        w = work(c)
        share = 6 if c["kind"] == "train" else (2 if c["D"] == 128 else 5)
        if w["flops"] <= limit["flops"] / share and w["bytes"] <= limit["bytes"]:
            return c


def _draw_once(rng):
    kind = rng.choice(["prefill", "prefill", "adaptive", "rows", "decode", "decode", "train", "layer"])
    D = 128 if kind in ("adaptive", "layer") else rng.choice(
        [64, 128, 128, 128] if kind == "train" else [64, 128, 128, 128, 256])
    H, Hkv = rng.choice([(8, 2), (16, 4), (16, 8)] if D != 128 else
                        [(32, 8), (32, 8), (40, 8), (16, 8), (8, 8), (32, 4)])
    c = dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp16"]), B=rng.choice([1, 1, 2]),
             H=H, Hkv=Hkv, D=D)
    if kind == "decode":
        dense = rng.random() < 0.5
        c.update(B=rng.choice([1, 1, 2, 7, 16, 32]), S=_log_int(rng, 300, 131072),
                 window=0 if dense else rng.choice([512, 1024, 2048, 4096]),
                 sink=0 if dense else rng.choice([64, 128, 1024]))
        return c
    if kind == "rows":
        n = _log_int(rng, 17, 2200)
        c.update(n=n, S=max(n, _log_int(rng, 600, 65536)))
        return c
    c.update(gamma=rng.choice([16, 32, 64, 64, 64, 128]),
             window=rng.choice([512, 1024, 2048, 2048, 4096]),
             sink=rng.choice([64, 128, 128, 1024]))
    if kind == "prefill":
        c.update(S=_log_int(rng, 600, 100000), mode=rng.choice(["delta", "delta", "delta", "recompute"]))
        if c["mode"] == "recompute":
            c["gamma"] = rng.choice([48, 64, 100])
    elif kind == "adaptive":
        c.update(B=1, S=_log_int(rng, 5000, 50000), gamma=64)
    elif kind == "train":
        c.update(S=64 * _log_int(rng, 10, 512))
    else:
        c.update(B=1, S=_log_int(rng, 300, 16000), H=32, Hkv=8, hidden=4096, inter=14336)
    return c


# ---------------------------------------------------------------------------
# inputs

def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _model_config(case):
    return LlamaConfig(vocab_size=1024, hidden_size=case.get("hidden", case["H"] * case["D"]),
                       intermediate_size=case.get("inter", 1024), num_hidden_layers=1,
                       num_attention_heads=case["H"], num_key_value_heads=case["Hkv"],
                       head_dim=case["D"], delta_lambda=case["gamma"],
                       sliding_window=case["window"], sink_tokens=case["sink"],
                       gamma_min=GAMMA_MIN, gamma_max=GAMMA_MAX, adapt_chunk=ADAPT_CHUNK,
                       stride_policy="adaptive" if case["kind"] == "adaptive" else "fixed")


def _layer(case, seed):
    with torch.device("cuda"):
        layer = LlamaDecoderLayer(_model_config(case), 0)
    layer = layer.to(DTYPES[case["dtype"]]).eval().requires_grad_(False)
    return init_weights_(layer, 0.02, seed)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dt, D, B, S = DTYPES[case["dtype"]], case["D"], case["B"], case["S"]
    kind = case["kind"]
    st = {"case": case, "scale": D ** -0.5}
    if kind == "layer":
        # hidden states of a mid-network residual stream, positions 0 .. S-1
        st["x"] = _randn(g, B, S, case["hidden"]).to(dt)
        pos = torch.arange(S, device="cuda")[None]
        cfg = _model_config(case)
        st["pe"] = rope_cos_sin(pos, D, cfg.rope_theta, dt, cfg.rope_scaling)
        st["layer"] = _layer(case, int(seed) + 1)
        return st
    n_q = {"decode": 1, "rows": case.get("n")}.get(kind, S)
    # caches keep room for the tokens to come
    n_kv = S + 128 if kind == "decode" else S
    st["q"] = _randn(g, B, n_q, case["H"], D).to(dt).transpose(1, 2)
    st["k"] = _randn(g, B, n_kv, case["Hkv"], D).to(dt)[:, :S].transpose(1, 2)
    st["v"] = _randn(g, B, n_kv, case["Hkv"], D).to(dt)[:, :S].transpose(1, 2)
    if kind == "rows":
        st["mask"] = torch.arange(S - n_q, S, device="cuda", dtype=torch.int64)[None]
    elif kind == "train":
        for t in ("q", "k", "v"):
            st[t].requires_grad_(True)
        st["up"] = _randn(g, B, S, case["H"], D).to(dt)
    elif kind == "adaptive":
        with torch.device("cuda"):
            st["module"] = LlamaAttention(_model_config(case), 0).to(dt).requires_grad_(False)
    return st


# ---------------------------------------------------------------------------
# one pass

def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "layer":
        with torch.no_grad():
            return st["layer"](st["x"], st["pe"])[0]
    q, k, v = st["q"], st["k"], st["v"]
    if kind == "prefill":
        return ops.delta_prefill(q, k, v, gamma=c["gamma"], window=c["window"], sink=c["sink"],
                                 sm_scale=st["scale"], mode=c["mode"])
    if kind == "adaptive":
        with torch.no_grad():
            return st["module"].delta_forward(st["module"], q, k, v, scaling=st["scale"])[0]
    if kind == "rows":
        return rows_attention(q, k, v, st["mask"], st["scale"])
    if kind == "decode":
        return ops.decode_attention(q, k, v, window=c["window"], sink=c["sink"], sm_scale=st["scale"])
    out = delta_forward_train(q, k, v, c["gamma"], c["window"], c["sink"])
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), st["up"]))


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _row_pairs(S, window, sink):
    """Visible keys of each row of key-sparse attention."""
    r = np.arange(S, dtype=np.int64)
    lo = np.maximum(r // Q_BLOCK * Q_BLOCK + Q_BLOCK - window, 0)
    return np.maximum(r - lo + 1, 0) + np.minimum(np.minimum(sink, r + 1), np.minimum(lo, r + 1))


def _attention_pairs(case, gamma=None):
    """(query, key) pairs per head of the delta composition: the key-sparse
    rows that are kept, and the causal rows of the anchors and the tail."""
    S, gamma = case["S"], gamma or case["gamma"]
    s_p = max(S - (S % gamma + max(128, gamma)), 0)
    sel = np.concatenate([np.arange(0, s_p, gamma), np.arange(s_p, S)])
    sp = _row_pairs(S, case["window"], case["sink"])
    sparse = sp[:s_p].sum()
    if case.get("mode") == "recompute":       # anchor rows are replaced
        sparse -= sp[sel[sel < s_p]].sum()
    return int(sparse) + int((sel + 1).sum())


def work(case):
    B, H, Hkv, D, S, kind = (case[x] for x in ("B", "H", "Hkv", "D", "S", "kind"))
    if kind == "decode":
        keys = S if case["window"] == 0 else min(S, case["window"] + case["sink"])
        return {"bytes": 2 * B * D * (2 * H + 2 * Hkv * keys), "flops": 4 * B * H * D * keys}
    if kind == "rows":
        n = case["n"]
        pairs = n * (S - n) + n * (n + 1) // 2
        return {"bytes": 2 * B * D * (2 * H * n + 2 * Hkv * S) + 8 * n, "flops": 4 * B * H * D * pairs}
    # the adaptive stride falls to its minimum on these inputs
    pairs = _attention_pairs(case, GAMMA_MIN if kind == "adaptive" else None)
    flops = 4 * B * H * D * pairs
    nbytes = 2 * B * S * D * (2 * H + 2 * Hkv)
    if kind == "train":      # five products backward for two forward
        return {"bytes": 2 * nbytes, "flops": flops * 7 // 2}
    if kind == "layer":
        weights = case["hidden"] * (2 * H * D + 2 * Hkv * D + 3 * case["inter"])
        return {"bytes": 2 * weights + 4 * B * S * case["hidden"], "flops": flops + 2 * B * S * weights}
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the present code differs from 64-bit arithmetic
    by (bf16: 0.0021-0.0034, gradients up to 0.0053, the decoder layer 0.0059;
    fp16: 0.0003-0.0004, gradients up to 0.0008): one rounding of the output
    plus those of the probabilities and of the branches that are summed."""
    rel = {"train": 2e-2, "layer": 2.4e-2}.get(case["kind"], 1.3e-2)
    return {"rel": rel if case["dtype"] == "bf16" else rel / 7}


# ---------------------------------------------------------------------------
# the same in plain torch at 64 bits

def _dense_rows(q, k, v, rows, scale, up=None):
    """Rows `rows` of q [B,H,S,D] against their causal keys -> [B,n,H,D]; with
    up [B,n,H,D] also the gradients of q's rows [B,n,H,D] and of k, v."""
    B, H, _, D = q.shape
    Hkv = k.shape[1]
    G = H // Hkv
    n = rows.numel()
    out = torch.empty(B, n, H, D, dtype=torch.float64, device=q.device)
    dq = torch.empty_like(out) if up is not None else None
    dk = torch.zeros_like(k) if up is not None else None
    dv = torch.zeros_like(v) if up is not None else None
    for b in range(B):
        for h in range(Hkv):
            hs = slice(h * G, (h + 1) * G)
            step = max(1, (1 << 28) // (G * k.shape[2]))
            for i in range(0, n, step):
                r = rows[i:i + step]
                m = int(r.max()) + 1
                kk, vv = k[b, h, :m].contiguous(), v[b, h, :m].contiguous()
                qr = q[b, hs][:, r].reshape(-1, D)
                s = qr @ kk.t().contiguous() * scale
                keys = torch.arange(m, device=q.device)
                s.view(G, -1, m).masked_fill_(keys > r[None, :, None], float("-inf"))
                p = torch.softmax(s, -1)
                o = p @ vv
                out[b, i:i + step, hs] = o.view(G, -1, D).transpose(0, 1)
                if up is not None:
                    do = up[b, i:i + step, hs].transpose(0, 1).reshape(-1, D)
                    dv[b, h, :m] += p.t().contiguous() @ do
                    ds = p * (do @ vv.t().contiguous() - (do * o).sum(-1, keepdim=True))
                    dq[b, i:i + step, hs] = (ds @ kk * scale).view(G, -1, D).transpose(0, 1)
                    dk[b, h, :m] += ds.t().contiguous() @ qr * scale
    return (out, dq, dk, dv) if up is not None else out


def _sparse_rows(q, k, v, window, sink, scale, up=None, step=512):
    """Key-sparse attention, every row -> [B,S,H,D]; with up [B,S,H,D] also
    the gradients of q [B,S,H,D], k and v."""
    B, H, S, D = q.shape
    Hkv = k.shape[1]
    G = H // Hkv
    out = torch.empty(B, S, H, D, dtype=torch.float64, device=q.device)
    dq = torch.empty_like(out) if up is not None else None
    dk = torch.zeros_like(k) if up is not None else None
    dv = torch.zeros_like(v) if up is not None else None
    for r0 in range(0, S, step):
        r1 = min(r0 + step, S)
        r = torch.arange(r0, r1, device=q.device)
        lo = r // Q_BLOCK * Q_BLOCK + Q_BLOCK - window
        first = max(int(lo[0]), 0)
        keys = torch.cat([torch.arange(0, min(sink, first, r1), device=q.device),
                          torch.arange(first, r1, device=q.device)])
        vis = (keys[None] <= r[:, None]) & ((keys[None] < sink) | (keys[None] >= lo[:, None]))
        for b in range(B):
            kk, vv = k[b][:, keys].contiguous(), v[b][:, keys].contiguous()
            qr = q[b, :, r0:r1].reshape(Hkv, G * (r1 - r0), D)
            s = torch.bmm(qr, kk.transpose(1, 2).contiguous()) * scale
            s.view(Hkv, G, r1 - r0, -1).masked_fill_(~vis, float("-inf"))
            # a row of a window shorter than its block may see no key at all
            p = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)
            o = torch.bmm(p, vv)
            out[b, r0:r1] = o.view(H, r1 - r0, D).transpose(0, 1)
            if up is not None:
                do = up[b, r0:r1].transpose(0, 1).reshape(Hkv, -1, D)
                dv[b][:, keys] += torch.bmm(p.transpose(1, 2).contiguous(), do)
                ds = p * (torch.bmm(do, vv.transpose(1, 2).contiguous()) - (do * o).sum(-1, keepdim=True))
                dq[b, r0:r1] = (torch.bmm(ds, kk) * scale).view(H, r1 - r0, D).transpose(0, 1)
                dk[b][:, keys] += torch.bmm(ds.transpose(1, 2).contiguous(), qr) * scale
    return (out, dq, dk, dv) if up is not None else out


def _selected(S, gamma, device):
    s_p = max(S - (S % gamma + max(128, gamma)), 0)
    return s_p, torch.cat([torch.arange(0, s_p, gamma, device=device),
                           torch.arange(s_p, S, device=device)])


def _delta_layer(q, k, v, case, scale):
    S, gamma = case["S"], case["gamma"]
    s_p, sel = _selected(S, gamma, q.device)
    out = _sparse_rows(q, k, v, case["window"], case["sink"], scale)
    dense = _dense_rows(q, k, v, sel, scale)
    n = sel.numel() - (S - s_p)
    if case.get("mode") == "recompute":
        out[:, sel] = dense
        return out
    if n:
        out[:, :s_p] += (dense[:, :n] - out[:, sel[:n]]).repeat_interleave(gamma, 1)[:, :s_p]
    out[:, s_p:] = dense[:, n:]
    return out


def _adaptive_layer(q, k, v, case, scale, threshold=0.95, margin=0.02):
    S = case["S"]
    s_p, _ = _selected(S, case["gamma"], q.device)
    out = _sparse_rows(q, k, v, case["window"], case["sink"], scale)
    gamma = case["gamma"]
    for a in range(0, s_p, ADAPT_CHUNK):
        e = min(a + ADAPT_CHUNK, s_p)
        idx = torch.arange(a, e, gamma, device=q.device)
        d = _dense_rows(q, k, v, idx, scale) - out[:, idx]
        cos = 1.0
        if idx.numel() > 1:
            cos = float(torch.nn.functional.cosine_similarity(d[:, 1:], d[:, :-1], dim=-1).mean())
        out[:, a:e] += d.repeat_interleave(gamma, 1)[:, :e - a]
        if cos < threshold:
            gamma = max(gamma // 2, GAMMA_MIN)
        elif cos > threshold + margin:
            gamma = min(gamma * 2, GAMMA_MAX)
    out[:, s_p:] = _dense_rows(q, k, v, torch.arange(s_p, S, device=q.device), scale)
    return out


def _train(q, k, v, up, case, scale):
    S, gamma = case["S"], case["gamma"]
    s_p, sel = _selected(S, gamma, q.device)
    n = sel.numel() - (S - s_p)
    up = up.double()
    dsp = up.clone()
    dsp[:, s_p:] = 0
    dd = up[:, s_p:]
    if n:
        da = up[:, :s_p].reshape(up.shape[0], n, gamma, *up.shape[2:]).sum(2)
        dsp[:, sel[:n]] -= da
        dd = torch.cat([da, dd], 1)
    out, dq, dk, dv = _sparse_rows(q, k, v, case["window"], case["sink"], scale, dsp)
    del dsp
    dense, eq, ek, ev = _dense_rows(q, k, v, sel, scale, dd)
    dq[:, sel] += eq
    if n:
        out[:, :s_p] += (dense[:, :n] - out[:, sel[:n]]).repeat_interleave(gamma, 1)
    out[:, s_p:] = dense[:, n:]
    return out, dq.transpose(1, 2), dk + ek, dv + ev


def _decoder_layer(st):
    case, layer, x = st["case"], st["layer"], st["x"].double()
    B, S, _ = x.shape
    cos, sin = (t.double()[:, :, None] for t in st["pe"])
    eps = layer.input_layernorm.variance_epsilon

    def norm(t, m):
        return m.weight.double() * t * torch.rsqrt(t.square().mean(-1, keepdim=True) + eps)

    def lin(t, m):
        return t @ m.weight.double().t()

    def rope(t):
        a, b = t.chunk(2, -1)
        return (t * cos + torch.cat((-b, a), -1) * sin).transpose(1, 2)

    at, mlp = layer.self_attn, layer.mlp
    h = norm(x, layer.input_layernorm)
    q, k, v = (lin(h, m).view(B, S, -1, case["D"]) for m in (at.q_proj, at.k_proj, at.v_proj))
    o = _delta_layer(rope(q), rope(k), v.transpose(1, 2), case, st["scale"])
    x = x + lin(o.reshape(B, S, -1), at.o_proj)
    h = norm(x, layer.post_attention_layernorm)
    return x + lin(torch.nn.functional.silu(lin(h, mlp.gate_proj)) * lin(h, mlp.up_proj), mlp.down_proj)


def exact(case, seed):
    st = prepare(case, seed)
    kind, scale = case["kind"], st["scale"]
    with torch.no_grad():
        if kind == "layer":
            return _decoder_layer(st)
        q, k, v = (st[t].detach().double() for t in ("q", "k", "v"))
        if kind == "prefill":
            return _delta_layer(q, k, v, case, scale)
        if kind == "adaptive":
            return _adaptive_layer(q, k, v, case, scale)
        if kind == "train":
            return _train(q, k, v, st["up"], case, scale)
        S = case["S"]
        if kind == "rows":
            qf = torch.zeros(case["B"], case["H"], S, case["D"], dtype=torch.float64, device=q.device)
            qf[:, :, S - case["n"]:] = q
            return _dense_rows(qf, k, v, torch.arange(S - case["n"], S, device=q.device), scale).transpose(1, 2)
        if case["window"] and case["window"] + case["sink"] < S:
            keep = torch.cat([torch.arange(case["sink"], device=q.device),
                              torch.arange(S - case["window"], S, device=q.device)])
            k, v = k[:, :, keep], v[:, :, keep]
        B, H, D = case["B"], case["H"], case["D"]
        G = H // case["Hkv"]
        s = (q.reshape(B, -1, G, D) @ k.transpose(2, 3).contiguous()) * scale
        return (torch.softmax(s, -1) @ v).reshape(B, H, 1, D)
