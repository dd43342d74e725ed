"""Single-token attention spread over several workgroups per (token, head):
the same key ranges, sums and order as one workgroup forms, so a decode step
of a few sequences (16 heads: 1, 2, 4 and 8 of them are spread over 16, 8, 4
and 2 workgroups) has the bits of a step of 16, which is not spread and which
test_gpu_attention.py pins to the oracle. Positions on both sides of the
spread's thresholds (256, 384, 512 keys) and of whole 32-key rounds, fewer than
16 ranges among them, up to the longest cache; one key dominates some
sequences."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import from_dev_bf16
from test_gpu_model import _build, _tiny_cfg

pytestmark = pytest.mark.gpu

POSITIONS = [511, 3499, 512, 4095, 255, 256, 257, 383, 384, 385, 300, 2048, 480, 3333, 1023, 1]


@pytest.mark.parametrize("nkv", [16, 4])
def test_spread_equals_single_workgroup(gpu, fmx, nkv):
    import torch
    from flashmlx_amd import model as M
    cfg = _tiny_cfg(num_attention_heads=16, num_key_value_heads=nkv, head_dim=128, max_position_embeddings=4096)
    n, max_seq = len(POSITIONS), 4096
    w, ref = _build(cfg, 51, n, max_seq, n)
    g = torch.Generator(device="cuda").manual_seed(52)
    k0, v0 = ref.kv_views()
    for c in (k0, v0):
        c.copy_(torch.randn(c.shape, generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16))
    k0[:, ::3, :, 0] *= 8.0
    past = [k0.clone(), v0.clone()]
    ids = torch.randint(0, cfg.vocab_size, (n, 1), generator=g, device="cuda", dtype=torch.int32)
    offs = torch.tensor(POSITIONS, dtype=torch.int32, device="cuda")
    logits = from_dev_bf16(ref.forward(ids, offs))
    hidden = from_dev_bf16(ref.hidden(n).clone())
    assert np.isfinite(ref.hidden(n).float().cpu().numpy()).all()
    for B in (1, 2, 4, 8):
        dm = M.DecoderModel(cfg, w, B, max_seq, B)
        for r in range(0, n, B):
            rows = slice(r, r + B)
            for _ in range(2):  # the arrival counts are back at zero
                for c, p in zip(dm.kv_views(), past):
                    c.copy_(p[:, rows])
                lg = from_dev_bf16(dm.forward(ids[rows], offs[rows].contiguous()))
                what = f"{B} sequences at {POSITIONS[rows]}"
                np.testing.assert_array_equal(from_dev_bf16(dm.hidden(B)), hidden[rows], err_msg=what)
                np.testing.assert_array_equal(lg, logits[rows], err_msg=what)
                for c, q in zip(dm.kv_views(), ref.kv_views()):
                    assert torch.equal(c.view(torch.int16), q[:, rows].contiguous().view(torch.int16)), what
