"""Blocks whose rows outgrow an XCD's L2 (4 MB): the static sets (shared
expert) then run an XCD's column groups over one pass before the next, in the
gate/up, relu^2 and down grids. A last pass of 53 rows and column groups that
the 8 XCDs do not share evenly (22 and 17; 11 and 17). Every row against the
same row of smaller forwards, which run every pass of one group first, and some
rows against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_close, assert_close_rows, from_dev_bf16, oracle_args, to_dev

pytestmark = pytest.mark.gpu

T, H, IS = 1525, 2176, 1408
PARTS = [(0, 700), (700, 1400), (T - 700, T)]
ROWS = np.array([0, 63, 64, 699, 1024, 1471, 1472, T - 1])


def test_block_rows_beyond_l2(gpu, fmx, oracle):
    from flashmlx_amd import workloads as W
    model = dict(W.QWEN15, hidden=H, n_experts=8, top_k=2, inter=256, shared_inter=IS)
    wl = W.Workload("rows_beyond_l2", model, T, 43)
    hi = W.host_inputs(wl)
    block, x = W.device_block(wl, hi)
    y = from_dev_bf16(block(x))
    for lo, hi_ in PARTS:
        np.testing.assert_array_equal(y[lo:hi_], from_dev_bf16(block(x[lo:hi_].contiguous())), err_msg=f"rows {lo}..")
    cfg, w = oracle_args(hi, model, oracle.quantize)
    ref, _, _ = oracle.moe_block(cfg, w, hi.x, oracle.ACC_A, tokens=ROWS)
    print(assert_close(y[ROWS], ref[ROWS], "rows beyond an L2"))


def test_nh_block_rows_beyond_l2(gpu, fmx, oracle):
    from flashmlx_amd import nemotron as N
    from flashmlx_amd.moe import synth_normal_bf16
    cfg = N.NhMoEConfig(hidden_size=H, n_routed_experts=16, num_experts_per_tok=4, moe_intermediate_size=256,
                        moe_shared_expert_intermediate_size=IS, routed_scaling_factor=2.5)
    w = N.synthetic_nh_weights(cfg, 44)
    x = synth_normal_bf16(T * H, 44, 7, 0.0, 1.0).reshape(T, H)
    block = N.NhMoEBlock(cfg, w, T)
    xd = to_dev(x)
    y = from_dev_bf16(block(xd))
    for lo, hi in PARTS:
        np.testing.assert_array_equal(y[lo:hi], from_dev_bf16(block(xd[lo:hi].contiguous())), err_msg=f"rows {lo}..")
    ref, _, _ = oracle.nh_moe_block(cfg.oracle_cfg(), N.host_weights(w), np.ascontiguousarray(x[ROWS]), oracle.ACC_F64)
    print(assert_close_rows(y[ROWS], ref, "rows beyond an L2"))


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_quantized_matmul_rows_beyond_l2(gpu, fmx, dtype):
    """One set alone, on both sides of the 512 work items from which it runs
    one pass after the other (45 column groups)."""
    import torch
    from flashmlx_amd import moe as Mo
    N, K = 5648, 2048
    dt = getattr(torch, dtype)
    g = torch.Generator(device="cuda").manual_seed(45)
    w = torch.randint(-2**31, 2**31, (N, K // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (torch.rand((N, K // 64), generator=g, device="cuda") * 0.01 + 0.002).to(dt)
    b = (torch.randn((N, K // 64), generator=g, device="cuda") * 0.05).to(dt)
    x = torch.randn((1105, K), generator=g, device="cuda").to(dt)
    y = Mo.quantized_matmul(x, w, s, b)
    for lo, hi in [(0, 600), (505, 1105), (1024, 1105)]:
        part = Mo.quantized_matmul(x[lo:hi].contiguous(), w, s, b)
        assert torch.equal(y[lo:hi].view(torch.int16), part.view(torch.int16)), f"rows {lo}.."
