"""Workloads of velograd_amd that its speed is judged on.

Each case is one call, or one forward and backward, of a layer through the entry points that a
model uses: the fused residual add + RMSNorm, its quantised outputs, the RMSNorm module, the rotary
embeddings and the norm + RoPE block input.  Sizes are those of the benchmark's configurations
(bench.py) and tests, and of generic hidden sizes around them.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, weights and modules on the GPU
    run(state)          one pass: its outputs
    work(case)          bytes and operations a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the same outputs in 64 bits, in plain torch
"""

import math

import torch

from velograd_amd import kernels, nn

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZES = {"fp32": 4, "fp16": 2, "bf16": 2}

# Kinds:
#   norm_fwd    kernels.fused_rmsnorm_residual_forward: inference, (y, h, inv_rms)
#   norm_fwdbwd the same and kernels.fused_rmsnorm_residual_backward on the saved h
#   norm_train  nn.FusedAddRMSNorm in a pre-norm block: gradients reach both y and h
#   module      nn.RMSNorm (no residual), forward and backward
#   fp8, mxfp8, mxfp4   the quantising forwards, for the next GEMM
#   rope        nn.apply_rope of q and k, forward and backward
#   rope_fwd    kernels.fused_rope of q and k (or of one tensor: kv_heads 0), inference
#   rotary      nn.apply_rotary_emb over the hidden vector, forward and backward
#   norm_rope   nn.RMSNormRoPE, the attention branch's input, forward and backward


def listed():
    return [
        # one decode step of a few sequences: latency and launches
        dict(name="decode_7x7168_bf16", kind="norm_fwd", batch=7, seq=1, dim=7168, dtype="bf16",
             eps=1e-6),
        # the smallest fp32 configuration: [4, 128, 768]
        dict(name="forward_4x128x768_fp32", kind="norm_fwd", batch=4, seq=128, dim=768,
             dtype="fp32", eps=1e-6),
        # a prefill of 8192 tokens
        dict(name="prefill_8192x4096_bf16", kind="norm_fwd", batch=1, seq=8192, dim=4096,
             dtype="bf16", eps=1e-5),
        # one training step of the block's norm on an ordinary micro-batch
        dict(name="train_1x2048x4096_bf16", kind="norm_train", batch=1, seq=2048, dim=4096,
             dtype="bf16", eps=1e-5),
        # the headline sizes as a model trains them: gradients through y and through h
        dict(name="train_8x2048x4096_bf16", kind="norm_train", batch=8, seq=2048, dim=4096,
             dtype="bf16", eps=1e-5),
        # the largest: forward and backward, activations with outliers
        dict(name="fwdbwd_32768x8192_bf16", kind="norm_fwdbwd", batch=1, seq=32768, dim=8192,
             dtype="bf16", eps=1e-5, outliers=True),
        # odd rows, which no 16- or 8-byte layout fits
        dict(name="fwdbwd_16384x4095_bf16", kind="norm_fwdbwd", batch=1, seq=16384, dim=4095,
             dtype="bf16", eps=1e-5),
        # quantised for an fp8 GEMM: one scale a row, prefill
        dict(name="fp8_16384x4096_bf16", kind="fp8", batch=1, seq=16384, dim=4096, dtype="bf16",
             eps=1e-5),
        # block-scaled fp4 at an in-between batch
        dict(name="mxfp4_257x7168_bf16", kind="mxfp4", batch=257, seq=1, dim=7168, dtype="bf16",
             eps=1e-6),
        # rotary embedding of one attention layer's q and k, training
        dict(name="rope_4x4096_32_8_128_bf16", kind="rope", batch=4, seq=4096, heads=32,
             kv_heads=8, head_dim=128, dtype="bf16", theta=5e5),
        # the reference benchmark's RoPE shape: one short fp32 tensor
        dict(name="rope_512x1024_64_fp32", kind="rope_fwd", batch=1, seq=512, heads=16, kv_heads=0,
             head_dim=64, dtype="fp32", theta=1e4),
        # the attention branch's input: norm and interleaved rotation, training
        dict(name="norm_rope_8x2048x4096_bf16", kind="norm_rope", batch=8, seq=2048, dim=4096,
             dtype="bf16", eps=1e-6, theta=1e4),
    ]


HIDDEN = (768, 1024, 1536, 2048, 3072, 4096, 5120, 6144, 7168, 8192, 12288, 16384)
KINDS = ("norm_fwd", "norm_fwd", "norm_fwd", "norm_fwdbwd", "norm_fwdbwd", "norm_train",
         "norm_train", "module", "fp8", "mxfp8", "mxfp4", "rope", "rope_fwd", "rotary",
         "norm_rope", "norm_rope")
MAX_TENSOR_BYTES = 256 << 20  # half of the largest listed case's


def draw(rng):
    kind = rng.choice(KINDS)
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
    tokens = int(round(2 ** rng.uniform(0, 15)))
    if kind in ("rope", "rope_fwd"):
        head_dim = rng.choice((64, 64, 80, 128, 128, 128, 256))
        heads = rng.choice((8, 16, 24, 32, 32, 40, 64))
        kv_heads = rng.choice((0, 1, heads // 8, heads // 4, heads))
        token_bytes = heads * head_dim * SIZES[dtype]
    else:
        if rng.random() < 0.3:  # ragged: odd ones among them, even where pairs or blocks ask it
            dim = int(round(2 ** rng.uniform(6, 13)))
            if kind in ("rotary", "norm_rope"):
                dim += dim % 2
            elif kind in ("mxfp8", "mxfp4"):
                dim = max(64, dim // 32 * 32)
        else:
            dim = rng.choice(HIDDEN)
        token_bytes = dim * SIZES[dtype]
    tokens = max(1, min(tokens, MAX_TENSOR_BYTES // token_bytes))
    batch = rng.choice((1, 1, 2, 4, 8))
    if kind in ("norm_fwd", "fp8", "mxfp8", "mxfp4") and tokens <= 512:
        batch, seq = tokens, 1  # decode: one token a sequence
    else:
        batch = min(batch, tokens)
        seq = tokens // batch
    case = dict(kind=kind, batch=batch, seq=seq, dtype=dtype)
    if kind in ("rope", "rope_fwd"):
        case.update(heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                    theta=rng.choice((1e4, 5e5)))
    else:
        case.update(dim=dim)
        if kind != "rotary":
            case.update(eps=rng.choice((1e-6, 1e-5)))
        if kind in ("rotary", "norm_rope"):
            case.update(theta=rng.choice((1e4, 5e5)))
        if kind in ("norm_fwd", "norm_fwdbwd", "norm_train") and dtype != "fp32":
            # weights kept in fp32 beside 16-bit activations: mixed-precision training
            case.update(fp32_weight=rng.random() < 0.25)
    return case


def _shapes(case):
    """The shapes of q and k (RoPE), or of the activations."""
    if case["kind"] in ("rope", "rope_fwd"):
        lead = (case["batch"], case["seq"])
        q = lead + (case["heads"], case["head_dim"])
        return q, (lead + (case["kv_heads"], case["head_dim"]) if case["kv_heads"] else None)
    return (case["batch"], case["seq"], case["dim"]), None


def _inputs(case, seed):
    """Activations and gradients ~ N(0, 1), or N(0, 2) with 0.1% of the entries 50 times as large;
    weights 1 + 0.1 N(0, 1)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    shape, k_shape = _shapes(case)

    def normal(size, scale=1.0):
        return torch.randn(size, generator=gen, device="cuda", dtype=dtype).mul_(scale)

    def activations(size):
        if not case.get("outliers"):
            return normal(size)
        t = normal(size, math.sqrt(2.0))
        n = t.numel() // 1000
        t.view(-1)[torch.randint(t.numel(), (n,), generator=gen, device="cuda")] *= 50
        return t

    kind = case["kind"]
    got = {"x": activations(shape)}
    if kind in ("rope", "rope_fwd"):
        got["k"] = normal(k_shape) if k_shape else None
        if kind == "rope":
            got["gx"] = normal(shape)
            got["gk"] = normal(k_shape) if k_shape else None
        return got
    if kind in ("norm_fwd", "norm_fwdbwd", "norm_train", "fp8", "mxfp8", "mxfp4"):
        got["res"] = activations(shape)
    if kind != "rotary":
        w = torch.randn(case["dim"], generator=gen, device="cuda").mul_(0.1).add_(1.0)
        got["w"] = w if case.get("fp32_weight") else w.to(dtype)
    if kind in ("norm_fwdbwd", "norm_train", "module", "rotary", "norm_rope"):
        got["gy"] = normal(shape)
    if kind == "norm_train":
        got["gh"] = normal(shape)
    return got


def prepare(case, seed):
    state = _inputs(case, seed)
    kind = case["kind"]
    state["case"] = case
    if kind in ("norm_train", "module", "norm_rope"):
        if kind == "norm_train":
            m = nn.FusedAddRMSNorm(case["dim"], eps=case["eps"])
        elif kind == "module":
            m = nn.RMSNorm(case["dim"], eps=case["eps"])
        else:
            m = nn.RMSNormRoPE(case["dim"], eps=case["eps"], base=case["theta"])
        m.weight = torch.nn.Parameter(state["w"])
        state["module"] = m
    if kind in ("norm_train", "module", "norm_rope", "rotary", "rope"):
        for name in ("x", "res", "k"):
            if state.get(name) is not None:
                state[name].requires_grad_(True)
    return state


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "norm_fwd":
        return kernels.fused_rmsnorm_residual_forward(x, state["res"], state["w"], case["eps"])
    if kind == "norm_fwdbwd":
        w = state["w"]
        y, h, inv_rms = kernels.fused_rmsnorm_residual_forward(x, state["res"], w, case["eps"])
        dx, dw = kernels.fused_rmsnorm_residual_backward(state["gy"], h, w, inv_rms,
                                                         saved_is_h=True)
        return y, h, inv_rms, dx, dw
    if kind == "norm_train":
        m, res = state["module"], state["res"]
        y, h = m(x, res)
        dx, dres, dw = torch.autograd.grad((y, h), (x, res, m.weight), (state["gy"], state["gh"]))
        return y, h, dx, dres, dw
    if kind in ("module", "norm_rope"):
        m = state["module"]
        y = m(x)
        dx, dw = torch.autograd.grad(y, (x, m.weight), state["gy"])
        return y, dx, dw
    if kind == "fp8":
        return kernels.fused_rmsnorm_residual_forward_fp8(x, state["res"], state["w"], case["eps"])
    if kind in ("mxfp8", "mxfp4"):
        fmt = "e4m3" if kind == "mxfp8" else "e2m1"
        q, scales, h, inv_rms = kernels.fused_rmsnorm_residual_forward_mx(
            x, state["res"], state["w"], case["eps"], fmt=fmt)
        return q.view(torch.uint8), scales.view(torch.uint8), h, inv_rms  # bytes for the GEMM
    if kind == "rotary":
        y = nn.apply_rotary_emb(x, case["theta"])
        return y, torch.autograd.grad(y, x, state["gy"])[0]
    k = state["k"]
    if kind == "rope_fwd":
        return kernels.fused_rope(x, k, base=case["theta"])
    q_rot, k_rot = nn.apply_rope(x, k, theta=case["theta"])
    if k is None:
        return q_rot, torch.autograd.grad(q_rot, x, state["gx"])[0]
    dq, dk = torch.autograd.grad((q_rot, k_rot), (x, k), (state["gx"], state["gk"]))
    return q_rot, k_rot, dq, dk


def work(case):
    kind, s = case["kind"], SIZES[case["dtype"]]
    rows = case["batch"] * case["seq"]
    if kind in ("rope", "rope_fwd"):
        n = rows * (case["heads"] + case["kv_heads"]) * case["head_dim"]
        passes = 2 if kind == "rope" else 1
        return {"bytes": passes * 2 * n * s, "flops": passes * 3 * n}
    d = case["dim"]
    n = rows * d
    if kind == "rotary":
        return {"bytes": 4 * n * s, "flops": 6 * n}
    w = d * (4 if case.get("fp32_weight") else s)
    stat = 4 * rows
    if kind == "norm_fwd":     # x, res, w in; y, h, inv_rms out
        return {"bytes": 4 * n * s + w + stat, "flops": 5 * n}
    if kind == "norm_fwdbwd":  # ... and g, h, w, inv_rms in; dx, dw out
        return {"bytes": 7 * n * s + 2 * w + 2 * stat + 4 * d, "flops": 14 * n}
    if kind == "norm_train":   # ... and grad_h in
        return {"bytes": 8 * n * s + 3 * w + 2 * stat, "flops": 15 * n}
    if kind == "module":       # x, w in; y, inv_rms out; then g, x, w, inv_rms in; dx, dw out
        return {"bytes": 5 * n * s + 3 * w + 2 * stat, "flops": 13 * n}
    if kind == "norm_rope":
        return {"bytes": 5 * n * s + 3 * w + 2 * stat, "flops": 19 * n}
    if kind == "fp8":          # x, res, w in; codes, scales, h, inv_rms out
        return {"bytes": 3 * n * s + n + w + 2 * stat, "flops": 7 * n}
    bytes_q = n if kind == "mxfp8" else n // 2
    return {"bytes": 3 * n * s + bytes_q + n // 32 + w + stat, "flops": 7 * n}


def tolerance(case):
    """About four times what the start's outputs are off the 64-bit ones: the rounding of the
    stored type (16 bits: 1.7e-3 bf16, 2.1e-4 fp16), or the fp32 sums' and angles' rounding."""
    kind, dtype = case["kind"], case["dtype"]
    if dtype == "bf16":
        t = {"rel": 7e-3, "max": 2e-2}
    elif dtype == "fp16":
        t = {"rel": 9e-4, "max": 3e-3}
    elif kind in ("rope", "rope_fwd"):
        # the angle is a float32 product: its rounding is position * 2^-24 radians at most
        t = {"rel": 2e-5, "max": 1e-3}
    else:
        t = {"rel": 3e-6, "max": 1e-4}
    if kind == "fp8":          # a code at a tie may fall to its neighbour, 1/8 of its value away
        t = {"rel": max(t["rel"], 2e-3), "max": 0.15}
    if kind in ("mxfp8", "mxfp4"):
        t["differ"] = 1e-3
    return t


def _rope_half(x, theta, sign):
    """The "rotate half" rotation with the angles that the entry point forms: float32 frequencies
    and products, then 64 bits."""
    seq, hd = x.shape[-3], x.shape[-1]
    half = hd // 2
    e = torch.arange(0, hd, 2, dtype=torch.float32, device=x.device) / hd
    freq = 1.0 / torch.pow(torch.tensor(theta, dtype=torch.float32, device=x.device), e)
    pos = torch.arange(seq, dtype=torch.float32, device=x.device)
    angle = torch.outer(pos, freq).double()[:, None, :]
    c, s = torch.cos(angle), torch.sin(angle) * sign
    x = x.double()
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, a * s + b * c), dim=-1)


def _rope_pairs(x, base, sign):
    """The interleaved rotation over the last axis, positions along axis -2, in 64 bits."""
    seq, d = x.shape[-2], x.shape[-1]
    freq = base ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    angle = torch.outer(torch.arange(seq, dtype=torch.float64, device=x.device), freq)
    c, s = torch.cos(angle), torch.sin(angle) * sign
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), dim=-1).flatten(-2)


def exact(case, seed):
    kind = case["kind"]
    v = _inputs(case, seed)
    if kind in ("rope", "rope_fwd"):
        theta = case["theta"]
        q = _rope_half(v["x"], theta, 1)
        k = _rope_half(v["k"], theta, 1) if v["k"] is not None else None
        if kind == "rope_fwd":
            return q if k is None else (q, k)
        dq = _rope_half(v["gx"], theta, -1)
        if k is None:
            return q, dq
        return q, k, dq, _rope_half(v["gk"], theta, -1)
    x = v["x"].double()
    if kind == "rotary":
        return (_rope_pairs(x, case["theta"], 1),
                _rope_pairs(v["gy"].double(), case["theta"], -1))
    w = v["w"].double()
    h = x + v["res"].double() if "res" in v else x
    mean_sq = h.square().mean(dim=-1, keepdim=True)
    inv = 1.0 / torch.sqrt(mean_sq.clamp(min=1e-12) + case["eps"])
    y = h * inv * w
    if kind == "norm_fwd":
        return y, h, inv
    if kind == "fp8":
        scale = y.abs().amax(dim=-1, keepdim=True) / 448.0
        codes = (y / scale).float().to(torch.float8_e4m3fn).double()
        return codes, scale, h, inv
    if kind in ("mxfp8", "mxfp4"):
        return None, None, h, inv
    g = v["gy"].double()
    if kind == "norm_rope":
        y = _rope_pairs(y, case["theta"], 1)
        g = _rope_pairs(g, case["theta"], -1)
    # the backward reads h as it is stored
    xhat = h.to(DTYPES[case["dtype"]]).double() * inv
    gw = g * w
    dx = inv * (gw - xhat * (gw * xhat).mean(dim=-1, keepdim=True))
    dw = (g * xhat).flatten(0, -2).sum(dim=0)
    if kind == "norm_fwdbwd":
        return y, h, inv, dx, dw
    if kind == "norm_train":
        dx = dx + v["gh"].double()
        return y, h, dx, dx, dw
    return y, dx, dw
