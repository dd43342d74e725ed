"""Attention of forwards with several tokens per sequence (causal, over the
KV cache, model.cpp:874-884) against fp64, at row and key counts around
multiples of 16 and 64, for MHA and GQA, head sizes on the matrix cores (64,
128) and off them (32): what the result is worth. That it has the oracle's
bits: test_gpu_attention_bits.py.

The decoder layer is built so that its residual stream is the attention's
output: no q projection (q is its bias, rotated), an identity o projection,
MoE experts that give zero, and an embedding of about 2^-12 (the input norm
scales it back up for k and v). Positions beyond the context hold NaN.

Tolerance: the output is rounded to bf16 twice (2^-9 of the value each, the
second with the embedding added, whose share is in the reference), and a
bf16 q from fp32 sines may round the other way in a few elements (2^-9 of
an element of q): scores up to about 10, whose relative error 2^-9 /
sqrt(hd) enters the weights, give at most 2^-9 of the largest value in the
weighted sum."""
from __future__ import annotations

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

V = 256
EPS = 1e-12


def _model(nh, nkv, hd, seed, B, max_seq, max_tokens):
    import torch
    from flashmlx_amd import model as M
    from flashmlx_amd.moe import MoEConfig, MoEWeights, QWeight, quantize
    H = nh * hd
    g = torch.Generator(device="cuda").manual_seed(seed)
    bf = torch.bfloat16

    def rnd(*s, std=1.0):
        return (torch.randn(s, generator=g, device="cuda") * std).to(bf)

    def const(rows, k, s):
        return QWeight(torch.zeros((*rows, k // 8), dtype=torch.int32, device="cuda"),
                       torch.full((*rows, k // 64), s, dtype=bf, device="cuda"),
                       torch.zeros((*rows, k // 64), dtype=bf, device="cuda"))

    moe = MoEConfig(hidden_size=H, num_experts=8, num_experts_per_tok=2, moe_intermediate_size=256,
                    shared_expert_intermediate_size=512, norm_topk_prob=False)
    cfg = M.ModelConfig(hidden_size=H, num_hidden_layers=1, num_attention_heads=nh, num_key_value_heads=nkv,
                        head_dim=hd, vocab_size=V, max_position_embeddings=4096, rms_norm_eps=EPS, moe=moe)
    eye = const((H,), H, 1.0)
    eye.w[torch.arange(H), torch.arange(H) // 8] = (1 << (4 * (torch.arange(H) % 8))).to(torch.int32).cuda()
    mw = MoEWeights(router_w=rnd(8, H, std=0.02), gate=const((8, 256), H, 0.0), up=const((8, 256), H, 0.0),
                    down=const((8, H), 256, 0.0))
    mw.shared_gate, mw.shared_up, mw.shared_down = const((512,), H, 0.0), const((512,), H, 0.0), const((H,), 512, 0.0)
    mw.shared_expert_gate_w = rnd(1, H, std=0.02)
    mw.pack(cfg.moe)
    kv = [QWeight(*quantize(rnd(nkv * hd, H, std=H ** -0.5))) for _ in range(2)]
    qb = rnd(nh * hd, std=2.0)
    lw = M.LayerWeights(input_norm_w=torch.ones(H, dtype=bf, device="cuda"),
                        post_norm_w=torch.ones(H, dtype=bf, device="cuda"),
                        qkv=M.pack_linear([const((nh * hd,), H, 0.0), *kv], H),
                        qkv_bias=torch.cat([qb, torch.zeros(2 * nkv * hd, dtype=bf, device="cuda")]),
                        o=M.pack_linear([eye], H), moe=mw)
    embed = rnd(V, H, std=2.0 ** -12)
    w = M.ModelWeights(embed=embed, norm_w=torch.ones(H, dtype=bf, device="cuda"),
                       lm_head=M.pack_linear([QWeight(*quantize(rnd(V, H, std=0.02)))], H), layers=[lw])
    dm = M.DecoderModel(cfg, w, B, max_seq, max_tokens)
    keys, values = dm.kv_views()
    keys.fill_(math.nan)
    values.fill_(math.nan)
    return cfg, w, dm, g


def _reference(cfg, w, dm, ids, pos):
    """embedding + attention in fp64 from the cached keys and values."""
    import torch
    nh, nkv, hd = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.hd
    B, L = ids.shape
    keys, values = dm.kv_views()
    q = w.layers[0].qkv_bias[:nh * hd].double().view(nh, hd)
    half = hd // 2
    inv = float(cfg.rope_theta) ** (-torch.arange(half, device="cuda", dtype=torch.float64) * 2 / hd)
    out = torch.empty((B, L, nh, hd), dtype=torch.float64, device="cuda")
    for b in range(B):
        p = pos[b] + torch.arange(L, device="cuda")
        th = p.double().unsqueeze(-1) * inv
        c, s = th.cos().float().double(), th.sin().float().double()
        n = int(p[-1]) + 1
        hide = torch.arange(n, device="cuda") > p.unsqueeze(-1)
        for h in range(nh):
            x1, x2 = q[h, :half], q[h, half:]
            qr = torch.cat([x1 * c - x2 * s, x1 * s + x2 * c], -1).to(torch.bfloat16).double()
            k, v = keys[0, b, h // (nh // nkv), :n].double(), values[0, b, h // (nh // nkv), :n].double()
            sc = (qr @ k.T.contiguous()) / math.sqrt(hd)
            # a hidden key's value does not count, whatever it is
            e = torch.softmax(sc.masked_fill(hide, -math.inf), -1)
            out[b, :, h] = torch.nan_to_num(e) @ torch.nan_to_num(v)
            bad = ~torch.isfinite(k).all(-1) | ~torch.isfinite(v).all(-1)
            out[b, (bad & ~hide).any(-1), h] = math.nan
    return w.embed[ids.reshape(-1).long()].double() + out.view(B * L, nh * hd)


def _check(cfg, w, dm, ids, offset, pos):
    import torch
    got = dm.forward(ids, offset, last_only=False)
    T = ids.numel()
    h = dm.hidden(T).double()
    ref = _reference(cfg, w, dm, ids, pos)
    torch.cuda.synchronize()
    assert got.shape[-1] == V
    nan = torch.isnan(ref)
    assert torch.equal(nan, ~torch.isfinite(h)), "rows that are not finite"
    tol = 2.0 ** -8 * ref.abs() + 2.0 ** -8 * ref[~nan].abs().max()
    err = (h - ref).abs().masked_fill(nan, 0)
    assert not (err > tol).logical_and(~nan).any(), (err.max(), ref[~nan].abs().max())
    rel = (err.square().sum() / ref[~nan].square().sum()).sqrt().item()
    assert rel < 2.0 ** -8, rel
    return rel


@pytest.mark.parametrize("nh,nkv,hd,B,L,ctx", [
    (4, 4, 128, 1, 2, 0), (4, 2, 128, 3, 48, 16), (4, 2, 128, 1, 2, 63), (4, 2, 128, 1, 17, 111), (4, 4, 128, 2, 65, 64),
    (8, 2, 128, 1, 130, 301), (8, 2, 64, 2, 33, 95), (8, 8, 64, 1, 300, 0), (16, 4, 128, 1, 1030, 0),
    (16, 16, 64, 1, 1025, 700), (32, 8, 64, 2, 257, 63), (4, 2, 32, 1, 40, 30)])
def test_attention_prefill(gpu, fmx, nh, nkv, hd, B, L, ctx):
    import torch
    max_seq = -(-(ctx + L + 3) // 64) * 64
    cfg, w, dm, g = _model(nh, nkv, hd, nh + L, B, max_seq, B * L)
    keys, values = dm.kv_views()
    for t in (keys, values):
        t[:, :, :, :ctx] = torch.randn(t[:, :, :, :ctx].shape, generator=g, device="cuda").to(torch.bfloat16)
    ids = torch.randint(0, V, (B, L), generator=g, device="cuda", dtype=torch.int32)
    print("relative error", _check(cfg, w, dm, ids, ctx, [ctx] * B))


def test_attention_prefill_sequence_offsets(gpu, fmx):
    """Several tokens per sequence at per-sequence device offsets."""
    import torch
    B, L, max_seq = 3, 37, 256
    cfg, w, dm, g = _model(4, 2, 128, 3, B, max_seq, B * L)
    pos = [0, 50, 170]
    keys, values = dm.kv_views()
    for b, p in enumerate(pos):
        for t in (keys, values):
            t[:, b, :, :p] = torch.randn(t[:, b, :, :p].shape, generator=g, device="cuda").to(torch.bfloat16)
    ids = torch.randint(0, V, (B, L), generator=g, device="cuda", dtype=torch.int32)
    _check(cfg, w, dm, ids, torch.tensor(pos, dtype=torch.int32, device="cuda"), pos)


@pytest.mark.parametrize("nh,L,bad_l", [(4, 50, 21), (16, 1030, 1001)])
def test_attention_prefill_not_finite(gpu, fmx, nh, L, bad_l):
    """A token whose embedding is infinite: its row and the later ones are
    NaN, the rows before it, also those in its tile, are not touched."""
    import torch
    cfg, w, dm, g = _model(nh, nh, 128, 5, 1, L + 2, L)
    w.embed[V - 1] = math.inf
    ids = torch.randint(0, V - 1, (1, L), generator=g, device="cuda", dtype=torch.int32)
    ids[0, bad_l] = V - 1
    _check(cfg, w, dm, ids, 0, [0])
