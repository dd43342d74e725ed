"""The lm_head of decode batches on the kernel for many tiles (1536 and more, for
up to 4 rows 2304; each workgroup several tiles) against the one-tile-per-workgroup kernel: every
logit is the same sum in the same order, so the logits of a vocabulary slice
have the bits of a model whose lm_head is that slice alone."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from helpers import from_dev_bf16
from test_gpu_model import _tiny_cfg

pytestmark = pytest.mark.gpu


# fewest tiles of the kernel (16 rows; up to 4 rows from 2304 tiles on), an
# uneven last round, one tile more; K of 4, 9 and 16 units (waves with one
# unit, with unequal ones, with four)
@pytest.mark.parametrize("V,H", [(1536 * 16, 512), (2305 * 16, 1152), (1537 * 16, 2048)])
def test_wide_lm_head_equals_slices(gpu, fmx, V, H):
    import torch
    from flashmlx_amd import model as M
    from flashmlx_amd.moe import QWeight, quantize
    cfg = _tiny_cfg(H=H, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=4, head_dim=64, vocab_size=512)
    w = M.synthetic_model(cfg, 61)
    g = torch.Generator(device="cuda").manual_seed(62)
    head = quantize((torch.randn((V, H), generator=g, device="cuda") * 0.02).to(torch.bfloat16))
    ids = torch.randint(0, 512, (16, 1), generator=g, device="cuda", dtype=torch.int32)
    for B in (1, 3, 16):
        for lo, hi in [(0, V), (0, 512), (V // 32 * 16, V // 32 * 16 + 512), (V - 512, V)]:
            c = dataclasses.replace(cfg, vocab_size=hi - lo)
            part = QWeight(*(t[lo:hi].contiguous() for t in head))
            dm = M.DecoderModel(c, dataclasses.replace(w, lm_head=M.pack_linear([part], H)), B, 16, B)
            lg = dm.forward(ids[:B], 0)
            assert torch.isfinite(lg).all()
            if hi - lo == V:
                whole = from_dev_bf16(lg)
            else:
                np.testing.assert_array_equal(whole[:, lo:hi], from_dev_bf16(lg),
                                              err_msg=f"{B} rows, columns {lo}:{hi}")
