"""The workloads by which this framework's speed is measured.

Each case is a call, or a training step, that a program makes of the framework's public entry points:
the FP8 and bf16 sliding-window attention, the FP8 linear layers in their three recipes with and
without the weight cache, the FP8 LM head, the FP8 decoder block in inference and the 450M decoder
block's training step. Sizes are those of the repository's workloads and tests, and generic ones
around them, down to a few tokens and with odd lengths. ``listed`` gives the fixed cases, ``draw``
more of the same ranges.

A case is a dict of plain values. ``prepare`` makes what the program has before the call (inputs,
layers, cached weight codes), ``run`` is one pass, ``work`` the bytes and operations a pass cannot do
without, ``tolerance`` how far two correct implementations may differ, and ``exact`` the same result
from plain torch in 64 bits (the e4m3 quantisation points of the recipes included: they are part of
what the operators compute).
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

E4M3_MAX = 448.0

# (in, out) widths of the linears of the two model sizes the framework is used with: d_model 1024
# with a 4096-wide MLP, and the 450M model's 1280 with a 3392-wide SwiGLU.
LINEARS = ((1024, 3072), (1024, 1024), (1024, 4096), (4096, 1024),
           (1280, 3840), (1280, 1280), (1280, 3392), (3392, 1280))
VOCAB = 16384


# ---------------------------------------------------------------------------------------- cases

def listed():
    return [
        # A short prompt through the FP8 attention: latency and launches.
        dict(name="attn_fp8_1k", kind="attn_fp8", B=1, H=8, T=1024, D=64, W=256, gran="head", packed=False),
        # The headline shape: long sequences, per-head scales.
        dict(name="attn_fp8_8k", kind="attn_fp8", B=4, H=16, T=8192, D=64, W=1024, gran="head", packed=False),
        # Wide heads, an odd length and window, one scale a tensor, q / k / v as the strided head
        # views of a fused projection's output.
        dict(name="attn_fp8_odd_d128", kind="attn_fp8", B=2, H=8, T=3001, D=128, W=777, gran="tensor", packed=True),
        # Training through the bf16 attention at the 450M model's shape.
        dict(name="attn_bf16_train_450m", kind="attn_bf16_train", B=2, H=20, T=8192, D=64, W=2048),
        # The same on a small ragged batch with wide heads.
        dict(name="attn_bf16_train_odd", kind="attn_bf16_train", B=1, H=8, T=1500, D=128, W=500),
        # Training through the FP8 attention, one 4096-token sequence of the 450M model.
        dict(name="attn_fp8_train_4k", kind="attn_fp8_train", B=1, H=20, T=4096, D=64, W=2048, gran="head"),
        # A few tokens through a linear whose codes are cached: serving.
        dict(name="linear_rowwise_16", kind="linear", recipe="rowwise", M=16, K=1024, N=4096),
        # An ordinary prompt through the weight-only linear.
        dict(name="linear_w8a16_200", kind="linear", recipe="weight_only", M=200, K=1280, N=3840),
        # A linear's training step (forward, dgrad, wgrad, weight quantised on the way).
        dict(name="linear_train_8k", kind="linear_train", recipe="tensorwise", M=8192, K=1024, N=4096),
        # Evaluation logits from the tied embedding, quantised on each call.
        dict(name="head_2k", kind="head", B=1, T=2047, K=1280, N=VOCAB),
        # A prompt through the whole FP8 decoder block with cached weights.
        dict(name="block_infer_2k", kind="block_infer", B=1, T=2048, W=1024),
        # The 450M block's training step, every gradient.
        dict(name="block_train_450m", kind="block_train", B=2, T=8192, W=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_attention(rng, kind):
    D = rng.choice((64, 64, 128, 32))
    while True:
        case = dict(kind=kind, B=rng.randint(1, 4), H=rng.choice((4, 8, 12, 16, 20)), T=_log_int(rng, 128, 8192), D=D,
                    W=_log_int(rng, 64, 4096))
        if case["B"] * case["H"] * case["T"] * min(case["W"], case["T"]) * D <= 2 * 20 * 8192 * 2048 * 64:
            break
    if kind != "attn_bf16_train":
        case["gran"] = rng.choice(("head", "head", "tensor", "bh"))
    if kind == "attn_fp8":
        case["packed"] = rng.random() < 0.5
    return case


def draw(rng):
    kind = rng.choice(("attn_fp8", "attn_fp8", "attn_bf16_train", "attn_bf16_train", "attn_fp8_train", "linear",
                       "linear", "linear", "linear_train", "linear_train", "head", "block_infer", "block_infer",
                       "block_train"))
    if kind.startswith("attn"):
        return _draw_attention(rng, kind)
    if kind in ("linear", "linear_train"):
        if rng.random() < 0.25:                      # other widths the conversion admits
            K, N = 64 * rng.randint(4, 64), 16 * rng.randint(16, 256)
        else:
            K, N = rng.choice(LINEARS)
        if kind == "linear":
            return dict(kind=kind, recipe=rng.choice(("rowwise", "tensorwise", "weight_only")),
                        M=_log_int(rng, 1, 16384), K=K, N=N)
        return dict(kind=kind, recipe=rng.choice(("rowwise", "tensorwise")), M=_log_int(rng, 64, 16384), K=K, N=N)
    if kind == "head":
        return dict(kind=kind, B=1, T=_log_int(rng, 16, 8192), K=rng.choice((1024, 1280)), N=VOCAB)
    if kind == "block_infer":
        return dict(kind=kind, B=1, T=_log_int(rng, 64, 32768), W=rng.choice((256, 1024, 2048, 4096)))
    return dict(kind="block_train", B=rng.randint(1, 2), T=_log_int(rng, 128, 8192), W=rng.choice((1024, 2048)))


# ---------------------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _heads(g, B, H, T, D):
    """Activations whose heads differ in scale, (B, H, T, D) fp32."""
    return _randn(g, B, H, T, D) * _randn(g, 1, H, 1, 1).exp()


def _qkv(case, g):
    B, H, T, D = (case[k] for k in "BHTD")
    if case["kind"] == "attn_fp8":
        qkv = [_heads(g, B, H, T, D).to(torch.bfloat16) for _ in range(3)]
    else:
        qkv = [_randn(g, B, H, T, D).to(torch.bfloat16) for _ in range(3)]
    if case.get("packed"):
        fused = torch.cat([t.transpose(1, 2).reshape(B, T, H * D) for t in qkv], dim=-1)
        qkv = [t.view(B, T, H, D).transpose(1, 2) for t in fused.chunk(3, dim=-1)]
    return qkv


def _rows(g, M, K):
    """Activation rows with one value in a thousand twenty times as large."""
    x = _randn(g, M, K)
    big = torch.rand(M, K, generator=g, device="cuda") < 1e-3
    return torch.where(big, x * 20.0, x).to(torch.bfloat16)


def _weight(g, N, K):
    return (_randn(g, N, K) * 0.02).to(torch.bfloat16)


def _fill_weights(module, g):
    """Every Linear weight ~ N(0, 0.02), every norm gain near 1."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.dim() == 2:
                p.copy_(_weight(g, *p.shape))
            else:
                p.copy_(1.0 + 0.1 * _randn(g, *p.shape))


def _linear_inputs(case, seed):
    g = _gen(seed)
    x, w = _rows(g, case["M"], case["K"]), _weight(g, case["N"], case["K"])
    dy = _randn(g, case["M"], case["N"]).to(torch.bfloat16) if case["kind"] == "linear_train" else None
    return x, w, dy


def _infer_block(case, g):
    from flower_amd.block import Fp8DecoderBlock
    with torch.device("cuda"):
        block = Fp8DecoderBlock(1024, 16, 4096, case["W"], max_seq_len=case["T"]).to(torch.bfloat16)
    _fill_weights(block, g)
    return block.eval()


def _train_block(case, g):
    from flower_amd.block import TransformerBlock, block_config
    from flower_amd.precision import convert_model_to_fp8
    with torch.device("cuda"):
        block = TransformerBlock(block_config(local_window=case["W"], max_seq_len=case["T"])).to(torch.bfloat16)
    _fill_weights(block, g)
    model = nn.Module()
    model.blocks = nn.ModuleList([block])
    convert_model_to_fp8(model, recipe="tensorwise", keep_bf16_blocks=0, verbose=False)
    return model.blocks[0]


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind.startswith("attn"):
        qkv = _qkv(case, g)
        state = dict(case=case, qkv=qkv)
        if kind != "attn_fp8":
            state["qkv"] = [t.requires_grad_(True) for t in qkv]
            state["do"] = _randn(g, *qkv[0].shape).to(torch.bfloat16)
        return state
    if kind in ("linear", "linear_train"):
        from flower_amd.precision import Fp8Linear, fp8_weight_cache
        x, w, dy = _linear_inputs(case, seed)
        lin = Fp8Linear(case["K"], case["N"], bias=False, device="cuda", dtype=torch.bfloat16, recipe=case["recipe"])
        with torch.no_grad():
            lin.weight.copy_(w)
        if kind == "linear_train":
            return dict(case=case, lin=lin, x=x.requires_grad_(True), dy=dy)
        cache = fp8_weight_cache(lin)
        cache.__enter__()
        return dict(case=case, lin=lin, cache=cache, x=x)
    if kind == "head":
        x = _randn(g, case["B"], case["T"], case["K"]).to(torch.bfloat16)
        return dict(case=case, x=x, w=_weight(g, case["N"], case["K"]))
    x = _randn(g, case["B"], case["T"], 1024 if kind == "block_infer" else 1280).to(torch.bfloat16)
    if kind == "block_infer":
        from flower_amd.precision import fp8_weight_cache
        block = _infer_block(case, g)
        cache = fp8_weight_cache(block)
        cache.__enter__()
        return dict(case=case, block=block, cache=cache, x=x)
    dy = _randn(g, *x.shape).to(torch.bfloat16)
    block = _train_block(case, g)
    return dict(case=case, block=block, x=x.requires_grad_(True), dy=dy, params=list(block.parameters()))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn_fp8":
        from flower_amd.kernels.fp8_swa_attention import fp8_swa_attention_forward
        return fp8_swa_attention_forward(*state["qkv"], case["W"], granularity=case["gran"])
    if kind == "attn_bf16_train":
        from flower_amd.kernels.swa_attention import swa_attention
        out = swa_attention(*state["qkv"], case["W"])
        return [out.detach(), *torch.autograd.grad(out, state["qkv"], state["do"])]
    if kind == "attn_fp8_train":
        from flower_amd.kernels.fp8_swa_attention import fp8_swa_attention
        out = fp8_swa_attention(*state["qkv"], case["W"], granularity=case["gran"])
        return [out.detach(), *torch.autograd.grad(out, state["qkv"], state["do"])]
    if kind == "linear":
        with torch.no_grad():
            return state["lin"](state["x"])
    if kind == "linear_train":
        y = state["lin"](state["x"])
        return [y.detach(), *torch.autograd.grad(y, [state["x"], state["lin"].weight], state["dy"])]
    if kind == "head":
        from flower_amd.precision import fp8_head
        with torch.no_grad():
            return fp8_head(state["x"], state["w"])
    if kind == "block_infer":
        return state["block"](state["x"])
    out = state["block"](state["x"])[0]
    return [out.detach(), *torch.autograd.grad(out, [state["x"], *state["params"]], state["dy"])]


# ---------------------------------------------------------------------------------------- work

def _pairs(T, W):
    W = min(W, T)
    return W * (W + 1) // 2 + (T - W) * W


def work(case):
    kind = case["kind"]
    if kind.startswith("attn"):
        B, H, T, D = (case[k] for k in "BHTD")
        n, pairs = B * H * T * D, B * H * _pairs(T, case["W"])
        if kind == "attn_fp8":                       # q, k, v -> out
            return dict(bytes=4 * 2 * n, flops=4 * D * pairs)
        return dict(bytes=8 * 2 * n, flops=14 * D * pairs)   # q, k, v, dout -> out, dq, dk, dv
    if kind in ("linear", "linear_train", "head"):
        M, K, N = case.get("M", case.get("T")), case["K"], case["N"]
        if kind == "linear":
            return dict(bytes=2 * M * K + N * K + 4 * N + 2 * M * N, flops=2 * M * N * K)
        if kind == "head":
            return dict(bytes=2 * M * K + 2 * N * K + 2 * M * N, flops=2 * M * N * K)
        return dict(bytes=4 * (M * K + N * K + M * N), flops=6 * M * N * K)
    B, T = case["B"], case["T"]
    if kind == "block_infer":
        d, weights = 1024, 1024 * (4 * 1024 + 2 * 4096)
        return dict(bytes=4 * B * T * d + weights, flops=2 * B * T * weights + 4 * d * B * _pairs(T, case["W"]))
    d, weights = 1280, 1280 * (4 * 1280 + 3 * 3392)
    return dict(bytes=8 * B * T * d + 4 * weights, flops=6 * B * T * weights + 14 * d * B * _pairs(T, case["W"]))


# ---------------------------------------------------------------------------------------- tolerance

# Measured against ``exact``: FP8 attention 0.003 - 0.037 (its e4m3 P), bf16 attention 0.0025, linears
# 0.0017 - 0.003 (the bf16 rounding of the results).

def tolerance(case):
    kind = case["kind"]
    if kind == "attn_fp8":           # e4m3 P: another block order rounds P to other codes
        return {"rel": 2e-2}
    if kind == "attn_bf16_train":    # bf16 P, dS and results
        return {"rel": 1e-2}
    if kind == "attn_fp8_train":
        return {"rel": 2e-2}
    if kind in ("linear", "linear_train", "head"):   # fp32 sums of the same codes, bf16 results
        return {"rel": 6e-3}
    # Whole blocks: a rounding shifts codes in the layers after it. Measured against ``exact``, whose
    # intermediate values are not rounded at all: 0.016 (inference), up to 0.054 (gradients).
    return {"rel": 6e-2 if kind == "block_train" else 3e-2}


# ---------------------------------------------------------------------------------------- 64-bit results

def _e4m3(x, dims, clamp=True):
    """x at its e4m3 codes and scale, the amax over ``dims`` (None: all), as float64."""
    x = x.float()
    amax = x.abs().amax() if dims is None else x.abs().amax(dim=dims, keepdim=True)
    s = amax.clamp_min(1e-12) / E4M3_MAX if clamp else (amax / E4M3_MAX).clamp_min(1e-12)
    q = x / s
    if clamp:
        q = q.clamp(-E4M3_MAX, E4M3_MAX)
    return q.to(torch.float8_e4m3fn).double() * s.double()


def _swa(q, k, v, W, do=None):
    """Causal sliding-window attention of (B, H, T, D) float64 tensors, a block of queries at a time;
    with ``do`` also its gradients."""
    B, H, T, D = q.shape
    out = torch.empty_like(q)
    if do is not None:
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    step = 512
    for b in range(B):
        for i0 in range(0, T, step):
            i1, j0 = min(i0 + step, T), max(0, i0 - W + 1)
            i = torch.arange(i0, i1, device=q.device)[:, None]
            j = torch.arange(j0, i1, device=q.device)[None, :]
            keep = (j <= i) & (i - j < W)
            qs, ks, vs = q[b, :, i0:i1], k[b, :, j0:i1], v[b, :, j0:i1]
            s = torch.matmul(qs, ks.transpose(-1, -2).contiguous()) / math.sqrt(D)
            p = torch.softmax(s.masked_fill_(~keep, float("-inf")), dim=-1)
            o = out[b, :, i0:i1] = torch.matmul(p, vs)
            if do is None:
                continue
            g = do[b, :, i0:i1]
            dv[b, :, j0:i1] += torch.matmul(p.transpose(-1, -2).contiguous(), g)
            dp = torch.matmul(g, vs.transpose(-1, -2).contiguous())
            ds = p.mul_(dp.sub_((g * o).sum(-1, keepdim=True))).div_(math.sqrt(D))
            dq[b, :, i0:i1] = torch.matmul(ds, ks)
            dk[b, :, j0:i1] += torch.matmul(ds.transpose(-1, -2).contiguous(), qs)
    return out if do is None else (out, dq, dk, dv)


class _SwaFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, W):
        ctx.save_for_backward(q, k, v)
        ctx.W = W
        return _swa(q, k, v, W)

    @staticmethod
    def backward(ctx, do):
        return (*_swa(*ctx.saved_tensors, ctx.W, do.contiguous())[1:], None)


class _TensorwiseFn(torch.autograd.Function):
    """y = x w^T with x, w and the gradient at their per-tensor e4m3 codes."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.shape = x.shape
        x2, w = _e4m3(x.reshape(-1, x.shape[-1]), None), _e4m3(w, None)
        ctx.save_for_backward(x2, w)
        return torch.matmul(x2, w.t().contiguous()).view(*x.shape[:-1], w.shape[0])

    @staticmethod
    def backward(ctx, g):
        x2, w = ctx.saved_tensors
        g2 = _e4m3(g.reshape(-1, g.shape[-1]), None)
        return torch.matmul(g2, w).view(ctx.shape), torch.matmul(g2.t().contiguous(), x2)


def _rms(x, eps=1e-6):
    return x * (x.pow(2).mean(-1, keepdim=True) + eps).rsqrt()


def _norm_heads_rope(y, H):
    """The q, k, v heads of a fused projection with QK-norm and RoPE (tables at their bf16 values)."""
    B, T, C = y.shape
    D = C // (3 * H)
    q, k, v = (t.reshape(B, T, H, D).transpose(1, 2) for t in y.chunk(3, dim=-1))
    inv = 1.0 / (10000.0 ** (torch.arange(0, D, 2).float() / D))
    ang = torch.outer(torch.arange(T).float(), inv)
    cos, sin = (t.repeat_interleave(2, dim=-1).to(y.device, torch.bfloat16).double() for t in (ang.cos(), ang.sin()))

    def rope(x):
        x = _rms(x)
        return x * cos + torch.stack((-x[..., 1::2], x[..., ::2]), dim=-1).flatten(-2) * sin

    return rope(q), rope(k), v


def _exact_attention(case, g):
    q, k, v = _qkv(case, g)
    W = case["W"]
    if case["kind"] == "attn_bf16_train":
        do = _randn(g, *q.shape).to(torch.bfloat16).double()
        return list(_swa(q.double(), k.double(), v.double(), W, do))
    dims = {"tensor": None, "head": (0, 2, 3), "bh": (2, 3)}[case["gran"]]
    q8, k8, v8 = (_e4m3(t, dims) for t in (q, k, v))
    if case["kind"] == "attn_fp8":
        return _swa(q8, k8, v8, W)
    # straight-through quantisers: the gradient is that of attention at the dequantised bf16 values
    do = _randn(g, *q.shape).to(torch.bfloat16).double()
    at = [t.to(torch.bfloat16).double() for t in (q8, k8, v8)]
    return [_swa(q8, k8, v8, W), *_swa(*at, W, do)[1:]]


def _exact_linear(case, seed):
    x, w, dy = _linear_inputs(case, seed)
    recipe = case["recipe"]
    if recipe == "tensorwise":
        ex, ew = _e4m3(x, None), _e4m3(w, None)
    else:
        ex = x.double() if recipe == "weight_only" else _e4m3(x, (1,), clamp=False)
        ew = _e4m3(w, (1,), clamp=False)
    y = torch.matmul(ex, ew.t().contiguous())
    if dy is None:
        return y
    if recipe == "tensorwise":
        eg = _e4m3(dy, None)
        return [y, torch.matmul(eg, ew), torch.matmul(eg.t().contiguous(), ex)]
    gx = torch.matmul(_e4m3(dy, (1,), clamp=False), _e4m3(w, (0,), clamp=False))
    gw = torch.matmul(_e4m3(dy, (0,), clamp=False).t().contiguous(), _e4m3(x, (0,), clamp=False))
    return [y, gx, gw]


def _exact_block_infer(case, g):
    x = _randn(g, case["B"], case["T"], 1024).to(torch.bfloat16)
    p = {n: t.detach() for n, t in _infer_block(case, g).named_parameters()}
    x = x.double()

    def linear(h, name):
        w = _e4m3(p[name + ".weight"], (1,), clamp=False)
        return torch.matmul(_e4m3(h, (-1,), clamp=False), w.t().contiguous())

    q, k, v = _norm_heads_rope(linear(_rms(x) * p["ln1.weight"].double(), "attn.qkv"), 16)
    a = _swa(*(_e4m3(t, (0, 2, 3)) for t in (q, k, v)), case["W"])
    x = x + linear(a.transpose(1, 2).reshape(x.shape), "attn.out")
    h = nn.functional.gelu(linear(_rms(x) * p["ln2.weight"].double(), "ff.net.0"))
    return x + linear(h, "ff.net.3")


def _exact_block_train(case, g):
    x = _randn(g, case["B"], case["T"], 1280).to(torch.bfloat16)
    dy = _randn(g, *x.shape).to(torch.bfloat16).double()
    p = {n: t.detach().double().requires_grad_(True) for n, t in _train_block(case, g).named_parameters()}
    x = x.double().requires_grad_(True)
    fp8 = _TensorwiseFn.apply
    q, k, v = _norm_heads_rope(fp8(_rms(x) * p["ln1.weight"], p["attn.qkv.weight"]), 20)
    a = _SwaFn.apply(q.contiguous(), k.contiguous(), v.contiguous(), case["W"])
    x1 = x + fp8(a.transpose(1, 2).reshape(x.shape), p["attn.out.weight"])
    h = _rms(x1) * p["ln2.weight"]
    h = nn.functional.silu(fp8(h, p["ff.gate.weight"])) * fp8(h, p["ff.up.weight"])
    out = x1 + fp8(h, p["ff.down.weight"])
    return [out.detach(), *torch.autograd.grad(out, [x, *p.values()], dy)]


def exact(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "block_train":
        return _exact_block_train(case, g)
    with torch.no_grad():
        if kind.startswith("attn"):
            return _exact_attention(case, g)
        if kind in ("linear", "linear_train"):
            return _exact_linear(case, seed)
        if kind == "head":
            x = _randn(g, case["B"], case["T"], case["K"]).to(torch.bfloat16)
            w = _e4m3(_weight(g, case["N"], case["K"]), (1,), clamp=False)
            return torch.matmul(_e4m3(x, (-1,), clamp=False), w.t().contiguous())
        return _exact_block_infer(case, g)
