"""The work that serving a 4-bit model has this package do, as cases that can be timed and checked.

A case is one pass through the public operators as a model's forward makes it: a single linear, the
linears of one decoder layer with their norms, or one mixture-of-experts feed-forward. The sizes are
those of the benchmark and of the reference's own measurements (hidden sizes 2048 to 8192, group
sizes 16 to 128, 128 experts with 8 per token), from one token of decode to a prefill of 8192.

kind "linear": y = x W^T through kernels.w4a8_linear.
kind "layer":  the norms and linears of one decoder layer at decode sizes: RMSNorm with its fp8 pair
               into qkv, o_proj, residual add + RMSNorm, fused gate_up + SiLU, down. Attention is not
               this package's: its output is an input of the case.
kind "moe":    route, grouped gate_up + SiLU, grouped down and the weighted sum through
               kernels.w4a8_moe.

fmt: "int4" (GPTQ symmetric), "awq" (int4 with zero points), "mxfp4", "nvfp4".
"""
from __future__ import annotations

import importlib

import torch

_PKG = "minisglang-rdna4_amd"
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16}
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)
_GROUP = {"mxfp4": 32, "nvfp4": 16}
_LARGEST_MACS = 8192 * 4096 * 28672
_LARGEST_MOE_MACS = 4096 * 8 * 3 * 2048 * 768


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # one token through one 4096 x 4096 projection: the smallest call a decode step makes
        dict(name="linear_m1_o_proj", kind="linear", fmt="int4", group=128, dtype="bf16", m=1, k=4096, n=4096),
        # one decode step of a Llama-3-8B-sized layer, GPTQ weights: five operators, one user
        dict(name="layer_m1_gptq", kind="layer", fmt="int4", group=128, dtype="bf16", m=1, hidden=4096, qkv=6144,
             attn=4096, inter=14336),
        # a batched decode step of a smaller AWQ model's layer in fp16 (9728 = its MLP width)
        dict(name="layer_m16_awq", kind="layer", fmt="awq", group=128, dtype="fp16", m=16, hidden=2560, qkv=6144,
             attn=4096, inter=9728),
        # a few users on the gate_up of a 70B-sized MXFP4 model
        dict(name="linear_m5_mxfp4", kind="linear", fmt="mxfp4", group=32, dtype="bf16", m=5, k=8192, n=28672),
        # a short prompt on the qkv projection
        dict(name="linear_m512_qkv", kind="linear", fmt="int4", group=128, dtype="bf16", m=512, k=4096, n=6144),
        # the largest call: a chunk of 8192 prompt tokens through gate_up
        dict(name="linear_m8192_gate_up", kind="linear", fmt="int4", group=128, dtype="bf16", m=8192, k=4096, n=28672),
        # a ragged prompt on AWQ weights with zero points, fp16
        dict(name="linear_m1777_awq", kind="linear", fmt="awq", group=128, dtype="fp16", m=1777, k=2560, n=9728),
        # GPTQ checkpoints with groups of 32 (the reference's own prefill shapes)
        dict(name="linear_m2048_g32", kind="linear", fmt="int4", group=32, dtype="fp16", m=2048, k=2816, n=2048),
        # MXFP4 prefill, the down projection of a 70B-sized model
        dict(name="linear_m4096_mxfp4", kind="linear", fmt="mxfp4", group=32, dtype="bf16", m=4096, k=28672, n=8192),
        # NVFP4 prefill
        dict(name="linear_m1024_nvfp4", kind="linear", fmt="nvfp4", group=16, dtype="bf16", m=1024, k=4096, n=14336),
        # batched decode of a 128-expert model: most of the time is reading the routed experts
        dict(name="moe_t16", kind="moe", fmt="int4", group=128, dtype="bf16", m=16, experts=128, top_k=8, hidden=2048,
             inter=768),
        # its prefill
        dict(name="moe_t4096", kind="moe", fmt="int4", group=128, dtype="bf16", m=4096, experts=128, top_k=8,
             hidden=2048, inter=768),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """lo..hi, uniform in the logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _multiple(rng, lo: int, hi: int, step: int) -> int:
    return max(1, _log_int(rng, lo, hi) // step) * step


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "layer", "moe"])
    fmt = rng.choice(["int4", "int4", "awq", "mxfp4", "nvfp4"])
    group = _GROUP.get(fmt) or rng.choice([128, 128, 64, 32])
    case = dict(kind=kind, fmt=fmt, group=group, dtype=rng.choice(["bf16", "fp16"]))
    if kind == "linear":
        case["m"] = _log_int(rng, 1, 8192)
        # most widths are multiples of 128; some only of the group
        case["k"] = _multiple(rng, 1024, 14336, rng.choice([128, 128, 128, max(group, 32)]))
        case["n"] = _multiple(rng, 1024, 28672, rng.choice([16, 128]))
        # the formats with narrow groups do more work per product
        most = _LARGEST_MACS // (4 if group < 128 and fmt != "mxfp4" else 1)
        while case["m"] * case["k"] * case["n"] > most:
            case["m"] = case["m"] * 3 // 4
    elif kind == "layer":
        case["m"] = _log_int(rng, 1, 16)
        case["hidden"] = _multiple(rng, 1024, 4096, 128)
        case["attn"] = _multiple(rng, 1024, 4096, 128)
        case["qkv"] = case["attn"] + 2 * 128 * rng.choice([2, 4, 8])
        case["inter"] = _multiple(rng, 2048, 14336, 128)
    else:
        case["m"] = _log_int(rng, 1, 4096)
        case["experts"] = rng.choice([32, 64, 96, 128])
        case["top_k"] = rng.choice([2, 4, 6, 8])
        case["hidden"] = _multiple(rng, 1024, 4096, 128)
        case["inter"] = _multiple(rng, 512, 1536, 128)
        while case["experts"] * case["hidden"] * case["inter"] > 128 * 2048 * 768:
            case["experts"] //= 2
        while case["m"] * case["top_k"] * 3 * case["hidden"] * case["inter"] > _LARGEST_MOE_MACS:
            case["m"] = case["m"] * 3 // 4
    return case


# ------------------------------------------------------------------------------------------------
# inputs, made on the GPU from the seed alone
# ------------------------------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(g, m: int, k: int, dtype) -> torch.Tensor:
    """N(0, 1) with one channel in a thousand 20 times as large, as a norm's output has them."""
    x = torch.randn(m, k, generator=g, device="cuda")
    idx = torch.randint(0, k, (max(1, k // 1000),), generator=g, device="cuda")
    x[:, idx] *= 20.0
    return x.to(dtype)


def _weight(g, n: int, k: int, fmt: str, group: int, lead: tuple = ()) -> dict:
    """Codes (*lead, n, k), group-major scales and, per format, zero points or the NVFP4 global, of a
    weight of about N(0, 0.02)."""
    dev = "cuda"
    w = dict(fmt=fmt, group=group)
    if fmt in ("int4", "awq"):
        w["codes"] = torch.randn(*lead, n, k, generator=g, device=dev).mul_(2.7).add_(8.0).round_().clamp_(0, 15).to(torch.uint8)
        w["scales"] = (0.0075 * (0.6 + 0.8 * torch.rand(*lead, k // group, n, generator=g, device=dev))).to(torch.float16)
        if fmt == "awq":
            w["zeros"] = torch.randint(5, 12, (*lead, k // group, n), generator=g, device=dev, dtype=torch.uint8)
        return w
    w["codes"] = torch.randint(0, 16, (*lead, n, k), generator=g, device=dev, dtype=torch.uint8)
    if fmt == "mxfp4":
        w["scales"] = torch.randint(119, 122, (*lead, k // 32, n), generator=g, device=dev, dtype=torch.uint8)
        return w
    w["scales"] = (torch.rand(*lead, k // 16, n, generator=g, device=dev) * 14.0 + 1.0).to(torch.float8_e4m3fn)
    w["global"] = (0.5 + torch.rand(*lead, n, generator=g, device=dev)) * 1e-3
    return w


def _pack8(codes: torch.Tensor) -> torch.Tensor:
    """(..., L) codes 0..15 -> (..., L/8) int32, code 8 i + j in nibble j of word i."""
    c = codes.view(*codes.shape[:-1], codes.shape[-1] // 8, 8)
    out = torch.zeros(c.shape[:-1], dtype=torch.int32, device=codes.device)
    for j in range(8):
        out |= c[..., j].to(torch.int32) << (4 * j)
    return out


def _op(w: dict) -> dict:
    """The operators' form of a weight: W4 tiles, scales and the zeros slot."""
    kernels = importlib.import_module(_PKG + ".quant.kernels")
    e2m1 = w["fmt"] in ("mxfp4", "nvfp4")
    zeros = None
    if "zeros" in w:
        zeros = _pack8(w["zeros"])
    elif "global" in w:
        zeros = w["global"].view(torch.int32)
    return dict(w=kernels.repack_w4(_pack8(w["codes"]), e2m1), s=w["scales"], z=zeros, group=w["group"], e2m1=e2m1)


def _inputs(case: dict, seed: int) -> dict:
    g, dt, fmt, grp, m = _gen(seed), _DT[case["dtype"]], case["fmt"], case["group"], case["m"]
    if case["kind"] == "linear":
        return dict(x=_activations(g, m, case["k"], dt), w=_weight(g, case["n"], case["k"], fmt, grp))
    h, i = case["hidden"], case["inter"]
    if case["kind"] == "layer":
        return dict(x=_activations(g, m, h, dt), attn=_activations(g, m, case["attn"], dt),
                    gain1=(1.0 + 0.1 * torch.randn(h, generator=g, device="cuda")).to(dt),
                    gain2=(1.0 + 0.1 * torch.randn(h, generator=g, device="cuda")).to(dt),
                    qkv=_weight(g, case["qkv"], h, fmt, grp), o=_weight(g, h, case["attn"], fmt, grp),
                    gate_up=_weight(g, 2 * i, h, fmt, grp), down=_weight(g, h, i, fmt, grp))
    e = case["experts"]
    return dict(x=_activations(g, m, h, dt), logits=torch.randn(m, e, generator=g, device="cuda").to(dt),
                w13=_weight(g, 2 * i, h, fmt, grp, (e,)), w2=_weight(g, h, i, fmt, grp, (e,)))


def prepare(case: dict, seed: int) -> dict:
    s = _inputs(case, seed)
    for name, v in s.items():
        if isinstance(v, dict):
            s[name] = _op(v)
    s["case"] = case
    s["kernels"] = importlib.import_module(_PKG + ".quant.kernels")
    if case["kind"] == "layer":
        norm = importlib.import_module(_PKG + ".layers.norm")
        for name in ("1", "2"):
            s["norm" + name] = norm.RMSNormFused(case["hidden"], 1e-6)
            s["norm" + name].weight = s.pop("gain" + name)
    return s


def run(state: dict):
    k, case = state["kernels"], state["case"]
    if case["kind"] == "linear":
        w = state["w"]
        return k.w4a8_linear(state["x"], w["w"], w["s"], w["z"], w["group"], weight_is_e2m1=w["e2m1"])
    if case["kind"] == "moe":
        a, b = state["w13"], state["w2"]
        return k.w4a8_moe(state["x"], a["w"], a["s"], a["z"], b["w"], b["s"], b["z"], state["logits"], case["top_k"],
                          True, weight_is_e2m1=a["e2m1"])
    q, o, gu, d = state["qkv"], state["o"], state["gate_up"], state["down"]
    h, _, xq, xs = state["norm1"].forward_quant(state["x"])
    qkv = k.w4a8_linear(h, q["w"], q["s"], q["z"], q["group"], weight_is_e2m1=q["e2m1"], x_fp8=xq, act_scales=xs)
    y = k.w4a8_linear(state["attn"], o["w"], o["s"], o["z"], o["group"], weight_is_e2m1=o["e2m1"])
    # the residual stream is x + y, held in y's storage from here on
    h2, res, _, _ = state["norm2"].forward_quant(state["x"], y)
    a = k.w4a8_linear_silu(h2, gu["w"], gu["s"], gu["z"], gu["group"], weight_is_e2m1=gu["e2m1"])
    out = k.w4a8_linear(a, d["w"], d["s"], d["z"], d["group"], weight_is_e2m1=d["e2m1"])
    return dict(qkv=qkv, residual=res, act=a, down=out)


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without, and what it gives in 64 bits
# ------------------------------------------------------------------------------------------------
def _weight_bytes(n: int, k: int, case: dict) -> float:
    fmt, g = case["fmt"], case["group"]
    per_group = {"int4": 2.0, "awq": 2.5, "mxfp4": 1.0, "nvfp4": 1.0}[fmt]
    return n * k / 2 + (k // g) * n * per_group + (4 * n if fmt == "nvfp4" else 0)


def work(case: dict) -> dict:
    m = case["m"]
    if case["kind"] == "linear":
        k, n = case["k"], case["n"]
        return dict(bytes=_weight_bytes(n, k, case) + 2 * m * (k + n), flops=2.0 * m * n * k)
    h, i = case["hidden"], case["inter"]
    if case["kind"] == "layer":
        mats = ((case["qkv"], h), (h, case["attn"]), (2 * i, h), (h, i))
        return dict(bytes=sum(_weight_bytes(n, k, case) for n, k in mats)
                    + 2 * m * (3 * h + case["attn"] + case["qkv"] + i) + 4 * h,
                    flops=2.0 * m * sum(n * k for n, k in mats))
    e, t = case["experts"], case["top_k"]
    read = e * (1.0 - (1.0 - t / e) ** m)  # experts that some token is routed to
    return dict(bytes=read * (_weight_bytes(2 * i, h, case) + _weight_bytes(h, i, case)) + 2 * m * (2 * h + e),
                flops=2.0 * m * t * 3 * h * i)


def tolerance(case: dict) -> dict:
    # one linear: sums in another order (the MFMA adds its 128 products in less than f32) move an output
    # across a rounding boundary of its type now and then. Measured between the decode and the tiled
    # kernels and against 64-bit sums rounded to the type: 2-norm 1.7e-4 for bf16 and 5.6e-5 for fp16,
    # a single value by one unit in the last place
    if case["kind"] == "linear":
        return dict(rel=7e-4, max=0.016) if case["dtype"] == "bf16" else dict(rel=2.5e-4, max=0.004)
    # several linears in a row: a rounding that flips is quantized to fp8 again for the next one, where
    # it may move by a whole step (3e-3 measured for the experts, 6e-3 for the down projection of a layer)
    return dict(rel=1.2e-2, max=0.24)


def _quantized(x: torch.Tensor) -> torch.Tensor:
    """x as per-token fp8 holds it: scale max(amax / 448, 1e-8), codes e4m3 to nearest even."""
    f = x.float()
    # by a tensor: a division by a Python number may become a multiplication by its reciprocal, and a
    # scale one unit off moves codes
    amax = f.abs().amax(dim=1, keepdim=True)
    s = (amax / torch.full_like(amax, 448.0)).clamp_min(1e-8)
    q = (f * torch.reciprocal(s)).to(torch.float8_e4m3fn)
    return q.double() * s.double()


def _dequantized(w: dict, e: int | None = None) -> torch.Tensor:
    pick = (lambda t: t) if e is None else (lambda t: t[e])
    codes, scales, fmt, g = pick(w["codes"]), pick(w["scales"]), w["fmt"], w["group"]
    if fmt in ("int4", "awq"):
        v = codes.double()
        s = scales.double()
        z = pick(w["zeros"]).double() if fmt == "awq" else torch.full_like(s, 8.0)
        v = v.view(v.shape[0], -1, g)
        return ((v - z.t().unsqueeze(-1)) * s.t().unsqueeze(-1)).reshape(codes.shape)
    v = torch.tensor(_E2M1, dtype=torch.float64, device=codes.device)[codes.long()]
    s = torch.exp2(scales.double() - 127.0) if fmt == "mxfp4" else scales.float().double() * pick(w["global"]).double()
    return (v.view(v.shape[0], -1, g) * s.t().unsqueeze(-1)).reshape(codes.shape)


def _silu_mul(y: torch.Tensor, dt) -> torch.Tensor:
    """silu(gate) * up of (m, 2 i), each step rounded to dt as the unfused pair rounds it."""
    gate, up = y.to(dt).double().chunk(2, dim=1)
    act = (gate / (1.0 + torch.exp(-gate))).to(dt).double()
    return (act * up).to(dt)


def _norm(x: torch.Tensor, gain: torch.Tensor) -> torch.Tensor:
    f = x.double()
    return (f * torch.rsqrt(f.square().mean(dim=1, keepdim=True) + 1e-6)).to(x.dtype) * gain


def exact(case: dict, seed: int):
    s, dt = _inputs(case, seed), _DT[case["dtype"]]
    if case["kind"] == "linear":
        return _quantized(s["x"]) @ _dequantized(s["w"]).t()
    if case["kind"] == "layer":
        qkv = _quantized(_norm(s["x"], s["gain1"])) @ _dequantized(s["qkv"]).t()
        y = (_quantized(s["attn"]) @ _dequantized(s["o"]).t()).to(dt)
        res = s["x"] + y
        a = _silu_mul(_quantized(_norm(res, s["gain2"])) @ _dequantized(s["gate_up"]).t(), dt)
        out = _quantized(a) @ _dequantized(s["down"]).t()
        return dict(qkv=qkv, residual=res.double(), act=a.double(), down=out)
    m, t = case["m"], case["top_k"]
    p = torch.softmax(s["logits"].double(), dim=1)
    w, ids = torch.sort(p, dim=1, descending=True, stable=True)  # ties go to the lower expert
    w, ids = w[:, :t], ids[:, :t]
    w = w / w.sum(dim=1, keepdim=True)
    x, y = _quantized(s["x"]), torch.zeros(m, t, case["hidden"], dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if tok.numel():
            a = _silu_mul(x[tok] @ _dequantized(s["w13"], e).t(), dt)
            y[tok, slot] = _quantized(a) @ _dequantized(s["w2"], e).t()
    return (y * w.unsqueeze(-1)).sum(dim=1)
