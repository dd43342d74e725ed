"""Performance cases of the framework: what a serving program calls, layer by
layer and as a whole, through the Python entry points.

Kinds of case:
  moe     MoEBlock calls, one per layer of a run of layers with weights of
          their own (a decode step walks through layers, so no layer finds
          its weights in a cache)
  nh      NhMoEBlock calls (Nemotron-H), the same way
  stack   one DecoderModel.forward: a prefill (length > 1, at a host offset)
          or a decode step (length 1, per-sequence device offsets)
  qmm     one quantized_matmul on MLX-layout weights
  gather  one gather_qmm on MLX-layout expert weights

Inputs are made by torch alone, from the seed: weights ~ N(0, 0.02)
quantized affine 4-bit in groups of 64, activations ~ N(0, 1) as a norm
leaves them. `exact` recomputes a case in 64 bits from the same inputs.
"""
from __future__ import annotations

import math

import torch

from flashmlx_amd import model as M
from flashmlx_amd import moe as Mo
from flashmlx_amd import nemotron as N

GROUP = 64
W_STD = 0.02
EPS, THETA = 1e-6, 1e6
HIDDEN, VOCAB, HEADS, HEAD_DIM = 2048, 151936, 16, 128

# the MoE layers of the shapes in flashmlx_amd/workloads.py and nemotron.py
MOE = {
    "qwen15": dict(E=60, k=4, I=1408, Is=5632, norm=False),
    "qwen3": dict(E=128, k=8, I=768, Is=0, norm=True),
}
NH = dict(H=2688, E=128, k=6, I=1856, Is=3712, scaling=2.5)


def listed():
    return [
        # interactive decoding of one sequence: the smallest call, latency
        dict(name="moe_qwen15_decode_1", kind="moe", model="qwen15", dtype="bf16", tokens=1, layers=8,
             bias=False, quant_router=False),
        # batched decoding, many experts in play
        dict(name="moe_qwen3_decode_8", kind="moe", model="qwen3", dtype="bf16", tokens=8, layers=4,
             bias=False, quant_router=False),
        # a short prompt of a float16 checkpoint with a quantized router
        dict(name="moe_qwen3_f16_100", kind="moe", model="qwen3", dtype="f16", tokens=100, layers=2,
             bias=False, quant_router=True),
        # an ordinary prompt, experts unevenly loaded
        dict(name="moe_qwen15_prefill_512", kind="moe", model="qwen15", dtype="bf16", tokens=512, layers=2,
             bias=True, quant_router=False),
        # a long prompt or several batched ones
        dict(name="moe_qwen15_prefill_4096", kind="moe", model="qwen15", dtype="bf16", tokens=4096, layers=1,
             bias=True, quant_router=False),
        # Nemotron-H: batched decoding and a prompt of odd length
        dict(name="nh_decode_4", kind="nh", tokens=4, layers=4),
        dict(name="nh_prefill_777", kind="nh", tokens=777, layers=1),
        # the stack: prefill of a long prompt of odd length
        dict(name="stack_prefill_3001", kind="stack", batch=1, length=3001, context=0, kv_heads=16, layers=2),
        # one sequence far into its context, and a decode batch of the server
        dict(name="stack_decode_1_at_3500", kind="stack", batch=1, length=1, context=3500, kv_heads=16, layers=4),
        dict(name="stack_decode_8_at_700", kind="stack", batch=8, length=1, context=700, kv_heads=16, layers=4),
        # the single operators on MLX arrays: the shared expert's projection
        # for a few rows, and the experts' for a prompt, in token order
        dict(name="qmm_45", kind="qmm", rows=45, n=5632, k=2048, dtype="bf16"),
        dict(name="gather_qmm_301", kind="gather", tokens=301, model="qwen15", dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "nh", "stack", "stack", "qmm", "gather"])
    if kind == "moe":
        T = _log_int(rng, 1, 4096)
        return dict(kind="moe", model=rng.choice(["qwen15", "qwen3"]), dtype=rng.choice(["bf16", "bf16", "f16"]),
                    tokens=T, layers=8 if T < 3 else 4 if T <= 16 else 2 if T <= 1024 else 1,
                    bias=rng.random() < 0.5, quant_router=rng.random() < 0.25)
    if kind == "nh":
        T = _log_int(rng, 1, 1500)
        return dict(kind="nh", tokens=T, layers=4 if T <= 16 else 1)
    if kind == "stack":
        kv = rng.choice([16, 16, 16, 4])
        if rng.random() < 0.5:
            return dict(kind="stack", batch=_log_int(rng, 1, 16), length=1, context=_log_int(rng, 16, 4000),
                        kv_heads=kv, layers=4)
        # a prompt, a batch of prompts, or a chunk that continues a context
        B = rng.choice([1, 1, 2, 4])
        L = _log_int(rng, 24, 3000 // B)
        ctx = 0 if rng.random() < 0.7 else _log_int(rng, 16, 1500)
        while ctx and B * L * (ctx + L // 2) > 4500000:  # no more than the longest listed prompt's attention
            ctx //= 2
        return dict(kind="stack", batch=B, length=L, context=ctx, kv_heads=kv, layers=2)
    if kind == "qmm":
        n, k = rng.choice([(5632, 2048), (2048, 5632), (2048, 2048)])
        return dict(kind="qmm", rows=_log_int(rng, 1, 4096), n=n, k=k, dtype=rng.choice(["bf16", "bf16", "f16"]))
    return dict(kind="gather", tokens=_log_int(rng, 1, 1024), model=rng.choice(["qwen15", "qwen3"]),
                dtype=rng.choice(["bf16", "bf16", "f16"]))


# ------------------------------------------------------------------ inputs

def _dt(case):
    return torch.float16 if case.get("dtype") == "f16" else torch.bfloat16


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))


def _randn(g, shape, std=1.0, dt=torch.bfloat16, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean).to(dt)


def _quantized(g, shape, dt=torch.bfloat16):
    """(words int32 [.., K/8], scales, biases [.., K/64]) of a N(0, 0.02) matrix."""
    *lead, K = shape
    rows = math.prod(lead)
    wq = torch.empty((rows, K // 8), dtype=torch.int32, device="cuda")
    sc = torch.empty((rows, K // GROUP), dtype=dt, device="cuda")
    bi = torch.empty_like(sc)
    step = max(1, (1 << 26) // K)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        w = torch.randn((n, K // GROUP, GROUP), generator=g, device="cuda", dtype=torch.float32).mul_(W_STD)
        lo, hi = torch.aminmax(w, dim=-1, keepdim=True)
        s, b = ((hi - lo) / 15).to(dt), lo.to(dt)
        q = w.sub_(b.float()).div_(s.float()).round_().clamp_(0, 15).to(torch.int32).view(n, K // 8, 8)
        word = q[..., 0].clone()
        for i in range(1, 8):
            word |= q[..., i] << (4 * i)
        wq[r:r + n], sc[r:r + n], bi[r:r + n] = word, s.view(n, -1), b.view(n, -1)
    return wq.view(*lead, K // 8), sc.view(*lead, K // GROUP), bi.view(*lead, K // GROUP)


def _moe_inputs(g, m, dt, bias, quant_router, H=HIDDEN):
    """One MoE layer's arrays."""
    E, I, Is = m["E"], m["I"], m["Is"]
    a = dict(gate=_quantized(g, (E, I, H), dt), up=_quantized(g, (E, I, H), dt), down=_quantized(g, (E, H, I), dt))
    a["router"] = _quantized(g, (E, H), dt) if quant_router else _randn(g, (E, H), W_STD, dt)
    a["bias"] = _randn(g, (E,), 1.0, dt) if bias else None
    if Is:
        a.update(sgate=_quantized(g, (Is, H), dt), sup=_quantized(g, (Is, H), dt), sdown=_quantized(g, (H, Is), dt))
        a["segate"] = _quantized(g, (1, H), dt) if quant_router else _randn(g, (1, H), W_STD, dt)
    return a


def _nh_inputs(g):
    H, E, I, Is = NH["H"], NH["E"], NH["I"], NH["Is"]
    return dict(gate_w=_randn(g, (E, H), W_STD), cbias=_randn(g, (E,), 0.05).float(), fc1=_quantized(g, (E, I, H)),
                fc2=_quantized(g, (E, H, I)), sup=_quantized(g, (Is, H)), sdown=_quantized(g, (H, Is)))


def _stack_inputs(case, g):
    H, hd, nkv = HIDDEN, HEAD_DIM, case["kv_heads"]
    B, L, ctx = case["batch"], case["length"], case["context"]
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(
            in_norm=_randn(g, (H,), 0.1, mean=1.0), post_norm=_randn(g, (H,), 0.1, mean=1.0),
            q=_quantized(g, (HEADS * hd, H)), k=_quantized(g, (nkv * hd, H)), v=_quantized(g, (nkv * hd, H)),
            o=_quantized(g, (H, HEADS * hd)), qkv_bias=_randn(g, ((HEADS + 2 * nkv) * hd,), 0.1),
            moe=_moe_inputs(g, MOE["qwen15"], torch.bfloat16, False, False)))
    a = dict(layers=layers, embed=_randn(g, (VOCAB, H), W_STD), norm=_randn(g, (H,), 0.1, mean=1.0),
             lm_head=_quantized(g, (VOCAB, H)))
    a["ids"] = torch.randint(0, VOCAB, (B, L), generator=g, device="cuda", dtype=torch.int32)
    # a server's sequences are at positions of their own
    back = torch.randint(0, max(1, ctx // 4), (B,), generator=g, device="cuda", dtype=torch.int32)
    a["offsets"] = (ctx - back) if L == 1 and B > 1 else torch.full((B,), ctx, dtype=torch.int32, device="cuda")
    # keys and values of the tokens before, of the size the projections give
    a["max_seq"] = min(4096, -(-(ctx + L + 1) // 64) * 64)
    a["k_past"] = _randn(g, (case["layers"], B, nkv, ctx, hd), 0.9)
    a["v_past"] = _randn(g, (case["layers"], B, nkv, ctx, hd), 0.9)
    return a


def _qw(t):
    return Mo.QWeight(*t)


def _opt_qw(t):
    return _qw(t) if isinstance(t, tuple) else t


def _moe_weights(a):
    w = Mo.MoEWeights(router_w=_opt_qw(a["router"]), gate=_qw(a["gate"]), up=_qw(a["up"]), down=_qw(a["down"]))
    w.router_logit_bias = a["bias"]
    if "sgate" in a:
        w.shared_gate, w.shared_up, w.shared_down = _qw(a["sgate"]), _qw(a["sup"]), _qw(a["sdown"])
        w.shared_expert_gate_w = _opt_qw(a["segate"])
    return w


def _moe_config(m, dt):
    return Mo.MoEConfig(hidden_size=HIDDEN, num_experts=m["E"], num_experts_per_tok=m["k"], moe_intermediate_size=m["I"],
                        shared_expert_intermediate_size=m["Is"], norm_topk_prob=m["norm"], activation_dtype=dt)


def _gather_inputs(case, g):
    m, dt = MOE[case["model"]], _dt(case)
    w = _quantized(g, (m["E"], m["I"], HIDDEN), dt)
    x = _randn(g, (case["tokens"], 1, 1, 1, HIDDEN), 1.0, dt)
    # every token's experts are distinct, some experts more popular than others
    pop = torch.randn((m["E"],), generator=g, device="cuda") * 0.5
    noise = torch.rand((case["tokens"], m["E"]), generator=g, device="cuda").clamp_min(1e-9)
    ids = (pop - torch.log(-torch.log(noise))).topk(m["k"], dim=-1).indices.to(torch.int32)
    return w, x, ids.view(case["tokens"], 1, m["k"]).contiguous()


def _qmm_inputs(case, g):
    return _quantized(g, (case["n"], case["k"]), _dt(case)), _randn(g, (case["rows"], case["k"]), 1.0, _dt(case))


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "moe":
        dt, m, T = _dt(case), MOE[case["model"]], case["tokens"]
        calls = []
        for _ in range(case["layers"]):
            w = _moe_weights(_moe_inputs(g, m, dt, case["bias"], case["quant_router"]))
            block = Mo.MoEBlock(_moe_config(m, dt), w, max_tokens=T)
            w.drop_mlx_layout()
            block.refresh()
            calls.append((block, _randn(g, (T, HIDDEN), 1.0, dt)))
        return dict(kind="blocks", calls=calls)
    if kind == "nh":
        calls = []
        for _ in range(case["layers"]):
            a = _nh_inputs(g)
            w = N.NhMoEWeights(gate_w=a["gate_w"], correction_bias=a["cbias"], fc1=_qw(a["fc1"]), fc2=_qw(a["fc2"]),
                               shared_up=_qw(a["sup"]), shared_down=_qw(a["sdown"]))
            block = N.NhMoEBlock(N.NhMoEConfig(), w, max_tokens=case["tokens"])
            w.drop_mlx_layout()
            calls.append((block, _randn(g, (case["tokens"], NH["H"]))))
        return dict(kind="blocks", calls=calls)
    if kind == "stack":
        a = _stack_inputs(case, g)
        cfg = M.ModelConfig(num_hidden_layers=case["layers"], num_key_value_heads=case["kv_heads"], head_dim=HEAD_DIM,
                            rms_norm_eps=EPS, rope_theta=THETA)
        layers = []
        for s in a["layers"]:
            mw = _moe_weights(s["moe"])
            mw.pack(cfg.moe)
            mw.drop_mlx_layout()
            layers.append(M.LayerWeights(
                input_norm_w=s["in_norm"], post_norm_w=s["post_norm"], qkv=M.pack_linear([_qw(s[n]) for n in "qkv"], HIDDEN),
                qkv_bias=s["qkv_bias"], o=M.pack_linear([_qw(s["o"])], HEADS * HEAD_DIM), moe=mw))
        w = M.ModelWeights(embed=a["embed"], norm_w=a["norm"], lm_head=M.pack_linear([_qw(a["lm_head"])], HIDDEN), layers=layers)
        B, L, ctx = case["batch"], case["length"], case["context"]
        dm = M.DecoderModel(cfg, w, B, a["max_seq"], B * L)
        keys, values = dm.kv_views()
        keys[:, :, :, :ctx] = a["k_past"]
        values[:, :, :, :ctx] = a["v_past"]
        return dict(kind="stack", model=dm, ids=a["ids"], offset=a["offsets"] if L == 1 else ctx)
    if kind == "qmm":
        w, x = _qmm_inputs(case, g)
        return dict(kind="qmm", w=w, x=x)
    w, x, ids = _gather_inputs(case, g)
    return dict(kind="gather", w=w, x=x, ids=ids)


def run(state):
    kind = state["kind"]
    if kind == "blocks":
        return [block(x) for block, x in state["calls"]]
    if kind == "stack":
        dm = state["model"]
        logits = dm.forward(state["ids"], state["offset"])
        keys, values = dm.kv_views()
        return dict(logits=logits, keys=keys, values=values)
    if kind == "qmm":
        return Mo.quantized_matmul(state["x"], *state["w"])
    return Mo.gather_qmm(state["x"], *state["w"], rhs_indices=state["ids"])


# ------------------------------------------------------------------ the work

def _wbytes(n, k):
    return n * k // 2 + 4 * n * (k // GROUP)


def _distinct(E, k, T):
    """Experts that T tokens' choices of k of E are expected to touch."""
    return E * (1.0 - (1.0 - k / E) ** T)


def _moe_work(m, T, quant_router=False, H=HIDDEN):
    E, k, I, Is = m["E"], m["k"], m["I"], m["Is"]
    byts = _distinct(E, k, T) * (2 * _wbytes(I, H) + _wbytes(H, I)) + (_wbytes(E, H) if quant_router else 2 * E * H)
    if Is:
        byts += 2 * _wbytes(Is, H) + _wbytes(H, Is)
    return byts + 4 * T * H, 2.0 * T * (3 * H * (k * I + Is) + H * E)


def work(case):
    kind = case["kind"]
    if kind == "moe":
        b, f = _moe_work(MOE[case["model"]], case["tokens"], case["quant_router"])
        return dict(bytes=b * case["layers"], flops=f * case["layers"])
    if kind == "nh":
        H, E, k, I, Is, T = NH["H"], NH["E"], NH["k"], NH["I"], NH["Is"], case["tokens"]
        b = _distinct(E, k, T) * (_wbytes(I, H) + _wbytes(H, I)) + 2 * E * H + _wbytes(Is, H) + _wbytes(H, Is) + 4 * T * H
        f = 2.0 * T * (2 * H * (k * I + Is) + H * E)
        return dict(bytes=b * case["layers"], flops=f * case["layers"])
    if kind == "stack":
        B, L, ctx, nkv, hd = case["batch"], case["length"], case["context"], case["kv_heads"], HEAD_DIM
        T, nqkv = B * L, (HEADS + 2 * case["kv_heads"]) * HEAD_DIM
        b, f = _moe_work(MOE["qwen15"], T)
        b += _wbytes(nqkv, HIDDEN) + _wbytes(HIDDEN, HEADS * hd) + B * nkv * hd * 4 * (ctx + 2 * L)
        f += 2.0 * T * HIDDEN * (nqkv + HEADS * hd) + 4.0 * B * HEADS * hd * L * (ctx + (L + 1) / 2)
        return dict(bytes=b * case["layers"] + _wbytes(VOCAB, HIDDEN) + 2 * T * HIDDEN + 2 * B * VOCAB,
                    flops=f * case["layers"] + 2.0 * B * VOCAB * HIDDEN)
    if kind == "qmm":
        T, n, k = case["rows"], case["n"], case["k"]
        return dict(bytes=_wbytes(n, k) + 2 * T * (n + k), flops=2.0 * T * n * k)
    m, T = MOE[case["model"]], case["tokens"]
    rows = T * m["k"]
    return dict(bytes=_distinct(m["E"], m["k"], T) * _wbytes(m["I"], HIDDEN) + 2 * T * HIDDEN + 2 * rows * m["I"] + 4 * rows,
                flops=2.0 * rows * m["I"] * HIDDEN)


def tolerance(case):
    kind = case["kind"]
    f16 = case.get("dtype") == "f16"
    # about four times what the path differs from the 64-bit result
    if kind in ("qmm", "gather"):
        # one product per output, rounded once (2^-9 bf16, 2^-12 float16),
        # with weights that may be rounded to float16 before it: 1.7e-3 bf16
        return dict(rel=2e-3, max=1e-2) if f16 else dict(rel=7e-3, max=2e-2)
    if kind == "moe":
        # two products with a rounding of the activations between them, and
        # scores and summands of the activation type: 5.5e-3 bf16, 7.4e-4 f16
        return dict(rel=3e-3, max=3e-2) if f16 else dict(rel=2e-2, max=0.15)
    if kind == "nh":
        return dict(rel=1.6e-2, max=0.12)  # 4e-3
    # whole layers, 1e-2 to 2.9e-2: a rounding may move an expert choice that
    # is nearly a tie
    return dict(rel=3e-2, max=0.9)


# ------------------------------------------------------------------ 64 bits

def _deq(t, i=None):
    """A quantized matrix [N, K] (expert i's) in float64."""
    w, s, b = t if i is None else (x[i] for x in t)
    q = (w.unsqueeze(-1) >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15
    q = q.reshape(w.shape[0], -1, GROUP).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(w.shape[0], -1)


def _row(t):
    return _deq(t) if isinstance(t, tuple) else t.double()


def _exact_moe(a, m, x, dt):
    """The MoE block: logits, probabilities and scores are values of the
    activation dtype by definition (the expert choice follows from them)."""
    x = x.double()
    logits = (x @ _row(a["router"]).T).to(dt)
    if a["bias"] is not None:
        logits = logits + a["bias"]
    probs = torch.softmax(logits.double(), -1).to(dt)
    scores, ids = torch.sort(probs, dim=-1, descending=True, stable=True)
    scores, ids = scores[:, :m["k"]], ids[:, :m["k"]]
    scores = scores.double()
    if m["norm"]:
        scores = scores / scores.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for e in range(m["E"]):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            xe = x[t]
            h = torch.nn.functional.silu(xe @ _deq(a["gate"], e).T) * (xe @ _deq(a["up"], e).T)
            y.index_add_(0, t, (h @ _deq(a["down"], e).T) * scores[t, slot].unsqueeze(-1))
    if "sgate" in a:
        h = torch.nn.functional.silu(x @ _deq(a["sgate"]).T) * (x @ _deq(a["sup"]).T)
        y += torch.sigmoid(x @ _row(a["segate"]).T) * (h @ _deq(a["sdown"]).T)
    return y


def _exact_nh(a, x):
    x = x.double()
    orig = torch.sigmoid((x @ a["gate_w"].double().T).to(torch.bfloat16).double())
    ids = torch.sort(orig.float() + a["cbias"], dim=-1, descending=True, stable=True).indices[:, :NH["k"]]
    scores = orig.gather(1, ids)
    scores = scores / scores.sum(-1, keepdim=True) * NH["scaling"]
    y = torch.zeros_like(x)
    for e in range(NH["E"]):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            h = torch.relu(x[t] @ _deq(a["fc1"], e).T).square()
            y.index_add_(0, t, (h @ _deq(a["fc2"], e).T) * scores[t, slot].unsqueeze(-1))
    return y + torch.relu(x @ _deq(a["sup"]).T).square() @ _deq(a["sdown"]).T


def _exact_norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _exact_rope(x, pos):
    """x [T, heads, hd] at positions pos [T]; pairs (i, i + hd / 2)."""
    half = HEAD_DIM // 2
    inv = THETA ** (-torch.arange(half, device="cuda", dtype=torch.float64) * 2 / HEAD_DIM)
    th = (pos.double().unsqueeze(-1) * inv).unsqueeze(1)
    c, s, x1, x2 = th.cos(), th.sin(), x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x1 * s + x2 * c], -1)


def _exact_stack(case, a):
    """The decoder in 64 bits; activations are kept as bf16 where a layer's
    inputs are defined as bf16 (what enters a norm, a projection, the cache)."""
    bf = lambda t: t.to(torch.bfloat16).double()  # noqa: E731
    B, L, ctx, nkv, hd = case["batch"], case["length"], case["context"], case["kv_heads"], HEAD_DIM
    T = B * L
    pos = (a["offsets"].long().unsqueeze(1) + torch.arange(L, device="cuda")).reshape(-1)
    seq = torch.arange(T, device="cuda") // L
    h = a["embed"][a["ids"].reshape(-1).long()].double()
    all_k = torch.zeros((case["layers"], B, nkv, a["max_seq"], hd), dtype=torch.float64, device="cuda")
    all_v = torch.zeros_like(all_k)
    all_k[:, :, :, :ctx], all_v[:, :, :, :ctx] = a["k_past"].double(), a["v_past"].double()
    for li, s in enumerate(a["layers"]):
        x = bf(_exact_norm(h, s["in_norm"]))
        w = torch.cat([_deq(s[n]) for n in "qkv"])
        qkv = bf(x @ w.T + s["qkv_bias"].double()).view(T, HEADS + 2 * nkv, hd)
        q = bf(_exact_rope(qkv[:, :HEADS], pos))
        keys, vals = all_k[li], all_v[li]
        keys[seq, :, pos] = _exact_rope(qkv[:, HEADS:HEADS + nkv], pos)
        vals[seq, :, pos] = qkv[:, HEADS + nkv:]
        kr = bf(keys)
        out = torch.empty((T, HEADS, hd), dtype=torch.float64, device="cuda")
        for b in range(B):
            rows = slice(b * L, (b + 1) * L)
            n = int(pos[rows].max()) + 1
            hide = torch.arange(n, device="cuda") > pos[rows].unsqueeze(-1)
            for hq in range(HEADS):
                g = hq // (HEADS // nkv)
                sc = (q[rows, hq] @ kr[b, g, :n].T.contiguous()) / math.sqrt(hd)
                out[rows, hq] = torch.softmax(sc.masked_fill_(hide, -math.inf), -1) @ vals[b, g, :n]
        h = bf(h + bf(out).view(T, -1) @ _deq(s["o"]).T)
        h = bf(h + _exact_moe(s["moe"], MOE["qwen15"], bf(_exact_norm(h, s["post_norm"])), torch.bfloat16))
    last = h.view(B, L, -1)[:, -1]
    x = bf(_exact_norm(last, a["norm"]))
    logits = torch.cat([x @ _deq(tuple(t[r:r + 16384] for t in a["lm_head"])).T for r in range(0, VOCAB, 16384)], -1)
    return dict(logits=logits, keys=all_k, values=all_v)


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "moe":
        dt, m, out = _dt(case), MOE[case["model"]], []
        for _ in range(case["layers"]):
            a = _moe_inputs(g, m, dt, case["bias"], case["quant_router"])
            out.append(_exact_moe(a, m, _randn(g, (case["tokens"], HIDDEN), 1.0, dt), dt))
        return out
    if kind == "nh":
        out = []
        for _ in range(case["layers"]):
            a = _nh_inputs(g)
            out.append(_exact_nh(a, _randn(g, (case["tokens"], NH["H"]))))
        return out
    if kind == "stack":
        return _exact_stack(case, _stack_inputs(case, g))
    if kind == "qmm":
        w, x = _qmm_inputs(case, g)
        return x.double() @ _deq(w).T
    w, x, ids = _gather_inputs(case, g)
    flat = ids.reshape(-1).long()
    xr = x.reshape(case["tokens"], HIDDEN).double().repeat_interleave(ids.shape[-1], 0)
    out = torch.empty((flat.numel(), w[0].shape[1]), dtype=torch.float64, device="cuda")
    for e in range(w[0].shape[0]):
        r = (flat == e).nonzero(as_tuple=True)[0]
        if r.numel():
            out[r] = xr[r] @ _deq(w, e).T
    return out.view(*ids.shape, 1, -1)
