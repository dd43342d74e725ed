"""quantized_matmul on the narrow column groups (few work items: 64 columns and
at most 32 rows each) against the wide ones: every output is the same sum in
the same order, so a few rows of a call have the bits they have among many."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


# one tile, a wave's tiles past the matrix, whole groups; K of one unit and of
# odd and even counts; rows around the passes; bf16 with a value outside
# fp16's range takes the exact arithmetic
@pytest.mark.parametrize("N,K", [(16, 128), (80, 640), (1024, 2048), (2064, 5632)])
@pytest.mark.parametrize("dtype,big", [("bfloat16", False), ("bfloat16", True), ("float16", False)])
def test_narrow_equals_wide(gpu, fmx, N, K, dtype, big):
    import torch
    from flashmlx_amd import moe as Mo
    dt = getattr(torch, dtype)
    g = torch.Generator(device="cuda").manual_seed(71)
    w = torch.randint(-2**31, 2**31, (N, K // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (torch.rand((N, K // 64), generator=g, device="cuda") * 0.01 + 0.002).to(dt)
    b = (torch.randn((N, K // 64), generator=g, device="cuda") * 0.05).to(dt)
    many = 32 * 512 // ((N // 16 + 3) // 4) + 33  # too many rows for the narrow groups
    x = torch.randn((many, K), generator=g, device="cuda").to(dt)
    if big:
        x[0, 5] = 1e6
    wide = Mo.quantized_matmul(x, w, s, b)
    q = ((w.unsqueeze(-1) >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15).reshape(N, K // 64, 64)
    deq = (q.double() * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(N, K)
    for rows in (1, 16, 17, 32, 33, 45, 64, 65):
        if dtype == "bfloat16" and rows < 32:
            continue  # another kernel
        y = Mo.quantized_matmul(x[:rows], w, s, b)
        assert torch.equal(y.view(torch.int16), wide[:rows].view(torch.int16)), f"{rows} rows"
        # one rounding to the output type, and weights rounded to fp16
        # (2^-11 of each, independently) before the products
        ref = x[:rows].double() @ deq.T
        err = (y.double() - ref).norm(dim=-1) / ref.norm(dim=-1)
        assert err.max().item() < (2 ** -8 if dtype == "bfloat16" else 2 ** -10), f"{rows} rows: {err.max().item()}"
