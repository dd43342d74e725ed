"""Attention of forwards with several tokens per sequence against the oracle
(orc_sdpa) bit for bit: scores in fp32 over d in order, weights and both sums
in fp64 over four key quarters, on the matrix cores (tiles of 16 rows and 16
keys, head sizes 64 and 128) as on the row kernel (head size 32, small calls).
Row and key counts on both sides of a tile and of the quarters, cached keys
whose scores grow with the position or a few of which dominate all others,
values near bf16's largest, scores that overflow, rows that are not finite.

The attention's output is read where the o projection takes it: in the
forward's workspace, behind the residual stream."""
from __future__ import annotations

import math

import numpy as np
import pytest

from helpers import bf16_to_f32, from_dev_bf16
from test_gpu_attention_prefill import V, _model

pytestmark = pytest.mark.gpu

P8 = [0, 4, 1, 5, 2, 6, 3, 7]  # the element in each slot of a run of 8


def _attention(cfg, dm, T):
    """(attention output, its fp16 copy in P8 order or None), [T, nh, hd]."""
    import torch
    H, nh, hd = cfg.hidden_size, cfg.num_attention_heads, cfg.hd
    off = dm.hidden(T).data_ptr() - dm.workspace.data_ptr()
    # the residual stream, the norm and its fp16 copy, q/k/v, rotated q
    for elems in (H, H, H, cfg.n_qkv, nh * hd):
        off += -(-T * elems * 2 // 256) * 256
    take = lambda o: dm.workspace[o:o + T * nh * hd * 2].view(torch.bfloat16)  # noqa: E731
    out = from_dev_bf16(take(off).clone()).reshape(T, nh, hd)
    if T <= 16:
        return out, None
    return out, from_dev_bf16(take(off + -(-T * nh * hd * 2 // 256) * 256).clone()).view(np.float16).reshape(T, nh, hd)


def _run(oracle, cfg, w, dm, ids, offset, pos):
    """One forward; its attention rows against the oracle: all of a short
    sequence, of a long one 40 at the start, at the end and between."""
    import torch
    nh, nkv, hd = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.hd
    B, L = ids.shape
    dm.forward(ids, offset, last_only=False)
    torch.cuda.synchronize()
    got, got_h = _attention(cfg, dm, B * L)
    got = got.reshape(B, L, nh, hd)
    if got_h is not None:
        f = bf16_to_f32(got).reshape(B * L, nh, hd // 8, 8)[..., P8].reshape(got_h.shape)
        with np.errstate(over="ignore"):
            same = (got_h == f.astype(np.float16)) | ~(np.abs(f) < 65504)
        assert same.all(), "fp16 copy"
    keys, values = (from_dev_bf16(t[0].contiguous()) for t in dm.kv_views())
    q0 = from_dev_bf16(w.layers[0].qkv_bias[:nh * hd].contiguous()).reshape(1, nh, hd)
    cs = oracle.rope_table(keys.shape[2], hd, float(cfg.rope_theta))
    scale = float(np.float32(1.0 / np.sqrt(hd)))
    n = L if L <= 320 else 40
    finite = 0
    for b in range(B):
        for s in sorted({min(s, L - n) for s in (0, 300, 500, 1010, L)}):
            q = oracle.rope(np.repeat(q0, n, axis=0), pos[b] + s + np.arange(n), cs)
            want = oracle.sdpa(q, keys[b], values[b], pos[b] + s, scale)
            fw, fg = bf16_to_f32(want), bf16_to_f32(got[b, s:s + n])
            bad = np.argwhere((got[b, s:s + n] != want) & ~(np.isnan(fw) & np.isnan(fg)))
            assert not bad.size, (f"sequence {b}, rows {s}..: {len(bad)} of {want.size} differ, first {bad[0]}: "
                                  f"{fg[tuple(bad[0])]} for {fw[tuple(bad[0])]}")
            finite += int(np.isfinite(fw).sum())
    return finite


def _past(dm, ctx, g):
    import torch
    return [torch.randn(t[:, :, :, :ctx].shape, generator=g, device="cuda") for t in dm.kv_views()]


def _set_past(dm, past, ctx):
    import torch
    for t, c in zip(dm.kv_views(), past):
        t[:, :, :, :ctx] = c.clamp(-3.3e38, 3.3e38).to(torch.bfloat16)


def _ids(g, B, L, hi=V):
    import torch
    return torch.randint(0, hi, (B, L), generator=g, device="cuda", dtype=torch.int32)


# few rows (rows x heads, by the caches' length): the row kernel; the others in tiles
@pytest.mark.parametrize("nh,nkv,hd,B,L,ctx", [
    (4, 4, 128, 1, 2, 0), (16, 16, 128, 1, 17, 111), (4, 2, 32, 1, 40, 30), (4, 4, 64, 2, 9, 60),
    (32, 8, 128, 13, 4, 0), (32, 8, 128, 13, 4, 61), (32, 8, 128, 9, 3, 260), (16, 2, 128, 3, 48, 16), (16, 16, 128, 1, 65, 64),
    (32, 4, 128, 1, 33, 4060), (8, 2, 128, 1, 130, 301), (16, 4, 128, 1, 1030, 0),
    (8, 2, 64, 6, 7, 500), (32, 2, 64, 5, 5, 95), (8, 8, 64, 1, 300, 0), (16, 16, 64, 1, 1025, 700), (32, 8, 64, 2, 257, 63)])
def test_attention_bits(gpu, fmx, oracle, nh, nkv, hd, B, L, ctx):
    cfg, w, dm, g = _model(nh, nkv, hd, nh + L, B, min(-(-(ctx + L + 3) // 64) * 64, 4096), B * L)
    _set_past(dm, _past(dm, ctx, g), ctx)
    _run(oracle, cfg, w, dm, _ids(g, B, L), ctx, [ctx] * B)


@pytest.mark.parametrize("nh,L", [(4, 37), (32, 37)])
def test_attention_bits_sequence_offsets(gpu, fmx, oracle, nh, L):
    """Several tokens per sequence at per-sequence device offsets."""
    import torch
    pos = [0, 50, 170]
    cfg, w, dm, g = _model(nh, 2, 128, 3, 3, 256, 3 * L)
    _set_past(dm, _past(dm, 170, g), 170)
    _run(oracle, cfg, w, dm, _ids(g, 3, L), torch.tensor(pos, dtype=torch.int32, device="cuda"), pos)


@pytest.mark.parametrize("nh,nkv,hd,B,L,ctx", [(16, 2, 128, 1, 70, 1100), (16, 4, 128, 1, 200, 700),
                                               (8, 2, 64, 1, 40, 530), (16, 16, 128, 18, 3, 1500)])
@pytest.mark.parametrize("kind", ["growing", "spikes", "ties", "large", "overflow"])
def test_attention_bits_extremes(gpu, fmx, oracle, nh, nkv, hd, B, L, ctx, kind):
    import torch
    cfg, w, dm, g = _model(nh, nkv, hd, 7, B, -(-(ctx + L + 3) // 64) * 64, B * L)
    past = _past(dm, ctx, g)
    q = w.layers[0].qkv_bias[:nh * hd].float().view(nkv, nh // nkv, hd)[:, 0]
    if kind == "growing":
        past[0] += q.view(1, 1, nkv, 1, hd) * torch.linspace(-1, 1, ctx, device="cuda").view(1, 1, 1, ctx, 1)
    elif kind == "spikes":  # in each quarter, first and last of a tile
        for p in (15, 16, ctx // 4, ctx // 2 - 1, ctx // 2, 3 * ctx // 4 + 17, ctx - 1):
            past[0][:, :, :, p] *= 3.0
    elif kind == "ties":
        # scores a rounding apart: for about half of the rows the key with the
        # largest exact sum is not the one with the largest fp32 score
        past[0][:] = past[0][:, :, :, :1]
        past[0][..., -32:] = torch.randn(past[0][..., -32:].shape, generator=g, device="cuda") * 2.0 ** -23
    elif kind == "large":
        past[1] *= 8e37
    else:  # sums of finite products: -inf for some rows, inf (then no weight is a number) for others
        past[0][:, :, :, ctx // 3] = 2.5e37 * torch.sign(q)
    _set_past(dm, past, ctx)
    _run(oracle, cfg, w, dm, _ids(g, B, L), ctx, [ctx] * B)


@pytest.mark.parametrize("nh,hd,L,bad_l", [(4, 128, 50, 21), (32, 128, 70, 21), (16, 64, 70, 21), (16, 128, 1030, 1001)])
def test_attention_bits_not_finite(gpu, fmx, oracle, nh, hd, L, bad_l):
    """A token whose embedding is infinite: its row and the later ones are
    NaN, the rows before it, also those in its tile, are not touched."""
    cfg, w, dm, g = _model(nh, nh, hd, 5, 1, L + 2, L)
    w.embed[V - 1] = math.inf
    ids = _ids(g, 1, L, V - 1)
    ids[0, bad_l] = V - 1
    assert _run(oracle, cfg, w, dm, ids, 0, [0]) > 0
