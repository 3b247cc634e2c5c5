"""The calls whose speed counts: a frozen quantized linear with its LoRA adapter, forward and backward, the fused
linears and producers of a Krea 2 block, and the quantization of a base weight.

Each case is a call a program makes through the package's modules: an image-generation loop runs the forwards without
gradients, a LoRA trainer runs forward and backward, and both quantize the base once when they start.  Every pass hands
the layer a tensor object that it has not seen (as each layer of a network does), so nothing computed for an earlier
pass's input is found again.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import __graft_entry__

k2 = __graft_entry__.load_package()

DEV = "cuda"
EPS = 1e-5                  # RMSNorm epsilon of the block
LARGEST = 1.3e12            # operations of the largest listed case's GEMM: no drawn case does more


# ---------------------------------------------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------------------------------------------
def _linear(name, base, tokens, k, n, rank, bias, train):
    c = {"kind": "linear", "base": base, "tokens": tokens, "in": k, "out": n, "rank": rank, "bias": bias, "train": train}
    return {"name": name, **c} if name else c


def listed():
    return [
        # adaLN modulation of a double-stream block at batch 2: one row per sample, the weight is streamed once
        _linear("adaln_w8", "w8a8", 2, 3072, 18432, 16, False, False),
        # a short prompt's text stream (its length is whatever the prompt gives), int4 base, generation
        _linear("text_w4", "w4a8", 333, 3072, 3072, 16, True, False),
        # text stream of 2 x 512 tokens through the MLP down-projection, generation with guidance
        _linear("text_down_w8", "w8a8", 1024, 12288, 3072, 16, False, False),
        # 4096 image tokens (1024 x 1024) through an attention projection, int4 base, fp32 bias
        _linear("image_w4", "w4a8", 4096, 3072, 3072, 16, True, False),
        # 2048 x 2048: 16384 image and 512 text tokens through the MLP up-projection, the largest forward
        _linear("up_2048_w8", "w8a8", 16896, 3072, 12288, 32, False, False),
        # LoRA training at 1024 x 1024 (4096 + 512 tokens) through the MLP down-projection, rank 64
        _linear("train_down_w8", "w8a8", 4608, 12288, 3072, 64, False, True),
        # LoRA training at 256 x 256 (256 + 512 tokens) through Krea 2's wq / gate / wo over an int4 base
        _linear("train_wo_w4", "w4a8", 768, 6144, 6144, 24, False, True),
        # the fp8 weight-only base at 1024 x 1024, generation, MLP gate / up of Krea 2
        _linear("up_fp8", "fp8", 4608, 6144, 16384, 16, False, False),
        # LoRA training over the fp8 base at 512 x 512 (1024 + 512 tokens) through Krea 2's wk / wv
        _linear("train_wk_fp8", "fp8", 1536, 6144, 1536, 32, False, True),
        # the modulated norm and the four linears that read it (wq, wk, wv, gate), generation at 1024 x 1024
        {"name": "attention_inputs", "kind": "attention", "batch": 1, "tokens": 4608, "width": 6144, "kv": 1536,
         "rank": 16, "train": False},
        # a whole MLP half of a block (modulated norm, gate / up, SwiGLU, down), LoRA training at 256 x 256, batch 1
        {"name": "train_mlp", "kind": "mlp", "batch": 1, "tokens": 768, "width": 6144, "hidden": 16384, "rank": 16,
         "train": True},
        # quantizing one bf16 MLP weight of Krea 2 to the fp8 base, as a trainer does for every weight at its start
        {"name": "quantize_fp8", "kind": "quantize", "base": "fp8", "in": 6144, "out": 16384, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi, step=1):
    return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))


def draw(rng):
    """One more call of the same ranges: tokens from one row to the 2048 x 2048 sequence, widths from the small test
    blocks' to Krea 2's, every base, ranks that do and do not fill the kernels' multiples of 16."""
    while True:
        kind = rng.choices(("linear", "attention", "mlp", "quantize"), (70, 10, 10, 10))[0]
        if kind == "linear":
            c = _linear(None, rng.choice(("w8a8", "w8a8", "w4a8", "fp8")), _log_int(rng, 1, 16896),
                        _log_int(rng, 512, 16384, 128), _log_int(rng, 512, 18432, 128),
                        rng.choice((4, 8, 16, 16, 24, 32, 64, 128)), rng.random() < 0.3, rng.random() < 0.4)
        elif kind == "attention":
            width = _log_int(rng, 1024, 6144, 256)
            batch = rng.choice((1, 2))
            c = {"kind": kind, "batch": batch, "tokens": batch * _log_int(rng, 64, 4608), "width": width,
                 "kv": max(256, width // 4 // 256 * 256), "rank": rng.choice((8, 16, 32)), "train": rng.random() < 0.5}
        elif kind == "mlp":
            width = _log_int(rng, 1024, 6144, 256)
            batch = rng.choice((1, 2))
            c = {"kind": kind, "batch": batch, "tokens": batch * _log_int(rng, 64, 2304), "width": width,
                 "hidden": width * 8 // 3 // 256 * 256, "rank": rng.choice((8, 16, 32)), "train": rng.random() < 0.5}
        else:
            c = {"kind": kind, "base": rng.choice(("w8a8", "w4a8", "fp8")), "in": _log_int(rng, 512, 16384, 128),
                 "out": _log_int(rng, 512, 18432, 128), "dtype": rng.choice(("bf16", "bf16", "f32"))}
        if work(c)["flops"] <= LARGEST:
            return c


# ---------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    t = torch.empty(shape, device=DEV, dtype=torch.float32).normal_(0.0, std, generator=g)
    return t.to(dtype)


def _activations(g, *shape):
    """N(0, 1) activations, 1 % of the channels 20 times as large (the outlier channels of a DiT)."""
    x = torch.empty(shape, device=DEV, dtype=torch.float32).normal_(generator=g)
    k = shape[-1]
    x[..., torch.randperm(k, device=DEV, generator=g)[:max(1, k // 100)]] *= 20.0
    return x.to(torch.bfloat16)


def _module(weight, bias=None):
    """An ``nn.Linear`` that holds the given tensors."""
    lin = nn.Linear(weight.shape[1], weight.shape[0], bias=bias is not None, device="meta")
    lin.weight = nn.Parameter(weight, requires_grad=False)
    if bias is not None:
        lin.bias = nn.Parameter(bias, requires_grad=False)
    return lin


def _linear_tensors(case, seed):
    g = _gen(seed)
    m, k, n, r = case["tokens"], case["in"], case["out"], case["rank"]
    t = {"x": _activations(g, m, k), "w": _normal(g, n, k, std=0.02),
         "A": _normal(g, r, k, std=0.01, dtype=torch.float32), "B": _normal(g, n, r, std=0.01, dtype=torch.float32)}
    t["bias"] = _normal(g, n, std=0.1, dtype=torch.float32) if case["bias"] else None
    if case["train"]:
        t["dy"] = _normal(g, m, n, std=1e-3)
    return t


def _parts(case):
    """The linears of a block case: (name, in, out)."""
    d = case["width"]
    if case["kind"] == "attention":
        return [("wq", d, d), ("wk", d, case["kv"]), ("wv", d, case["kv"]), ("gate", d, d)]
    return [("gate", d, case["hidden"]), ("up", d, case["hidden"]), ("down", case["hidden"], d)]


def _block_tensors(case, seed):
    g = _gen(seed)
    d, r = case["width"], case["rank"]
    shape = (case["batch"], case["tokens"] // case["batch"])
    t = {"x": _normal(g, *shape, d), "norm": _normal(g, d, std=0.1, dtype=torch.float32),
         "scale": _normal(g, case["batch"], 1, d, std=0.3), "shift": _normal(g, case["batch"], 1, d, std=0.3)}
    for name, k, n in _parts(case):
        t["w." + name] = _normal(g, n, k, std=0.02)
        t["A." + name] = _normal(g, r, k, std=0.01, dtype=torch.float32)
        t["B." + name] = _normal(g, n, r, std=0.01, dtype=torch.float32)
    if case["train"]:
        outs = _parts(case) if case["kind"] == "attention" else _parts(case)[-1:]
        t["dy"] = [_normal(g, *shape, n, std=1e-3) for _, _, n in outs]
    return t


class _Norm(nn.Module):
    def __init__(self, scale):
        super().__init__()
        self.eps = EPS
        self.scale = nn.Parameter(scale, requires_grad=False)


class _Holder(nn.Module):
    pass


def prepare(case, seed):
    if case["kind"] == "quantize":
        w = _normal(_gen(seed), case["out"], case["in"], std=0.02,
                    dtype=torch.bfloat16 if case["dtype"] == "bf16" else torch.float32)
        return {"case": case, "lin": _module(w)}
    if case["kind"] == "linear":
        t = _linear_tensors(case, seed)
        lin = _module(t["w"], t["bias"])
        base = k2.Fp8Linear(lin) if case["base"] == "fp8" else k2.ConvRotLinear(lin, case["base"])
        layer = k2.LoRALinear(base, case["rank"], float(case["rank"]))
        with torch.no_grad():
            layer.lora_A.copy_(t["A"])
            layer.lora_B.copy_(t["B"])
        return {"case": case, "layer": layer, "x": t["x"], "dy": t.get("dy")}
    t = _block_tensors(case, seed)
    dit, block, part = _Holder(), _Holder(), _Holder()
    where = "attn" if case["kind"] == "attention" else "mlp"
    for name, _, _ in _parts(case):
        setattr(part, name, _module(t["w." + name]))
    setattr(block, where, part)
    dit.blocks = nn.ModuleList([block])
    k2.quantize_dit_convrot(dit, "w8a8")
    k2.inject_lora(dit, case["rank"])
    k2.group_siblings(dit)
    layers = [getattr(part, name) for name, _, _ in _parts(case)]
    with torch.no_grad():
        for (name, _, _), layer in zip(_parts(case), layers):
            layer.lora_A.copy_(t["A." + name])
            layer.lora_B.copy_(t["B." + name])
    return {"case": case, "layers": layers, "norm": _Norm(t["norm"]), "x": t["x"], "scale": t["scale"],
            "shift": t["shift"], "dy": t.get("dy")}


# ---------------------------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------------------------
def _block_forward(s, x):
    h = k2.modulated_rmsnorm(s["norm"], x, s["scale"], s["shift"])
    if s["case"]["kind"] == "attention":
        return [layer(h) for layer in s["layers"]]
    gate, up, down = s["layers"]
    return [down(k2.swiglu(gate(h), up(h)))]


def run(s):
    case = s["case"]
    if case["kind"] == "quantize":
        if case["base"] == "fp8":
            q = k2.Fp8Linear(s["lin"])
            return [q.weight_fp8.data.view(torch.uint8), q.scale.data.view(torch.int16)]
        q = k2.ConvRotLinear(s["lin"], case["base"])
        return [q.qweight.data, q.wscale.data]
    layers = [s["layer"]] if case["kind"] == "linear" else s["layers"]

    def forward(x):
        return [layers[0](x)] if case["kind"] == "linear" else _block_forward(s, x)

    if not case["train"]:
        with torch.no_grad():
            return forward(s["x"].detach())
    x = s["x"].detach().requires_grad_()
    ys = forward(x)
    adapters = [p for layer in layers for p in (layer.lora_A, layer.lora_B)]
    grads = torch.autograd.grad(ys, [x, *adapters], [s["dy"]] if case["kind"] == "linear" else s["dy"])
    return [y.detach() for y in ys] + list(grads)


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without, and what it may differ by
# ---------------------------------------------------------------------------------------------------------------
_WBYTES = {"w8a8": 1.0, "w4a8": 0.5 + 2 / 64, "fp8": 1.0}


def work(case):
    if case["kind"] == "quantize":
        size = case["in"] * case["out"]
        return {"bytes": size * ((2 if case["dtype"] == "bf16" else 4) + _WBYTES[case["base"]]), "flops": 16.0 * size}
    m = case["tokens"]
    parts = [("", case["in"], case["out"])] if case["kind"] == "linear" else _parts(case)
    r = case["rank"]
    weights = sum(k * n for _, k, n in parts) * _WBYTES[case.get("base", "w8a8")]
    factors = sum(4 * r * (k + n) for _, k, n in parts)
    k_in = case["in"] if case["kind"] == "linear" else case["width"]
    n_out = sum(n for _, _, n in parts) if case["kind"] != "mlp" else case["width"]
    nbytes = weights + factors + 2 * m * (k_in + n_out)
    flops = sum(2.0 * m * n * k + 2.0 * m * r * (k + n) for _, k, n in parts)
    if case["train"]:          # the output gradient in, the input gradient and the factors' gradients out
        nbytes += 2 * m * (k_in + n_out) + factors
        flops += sum(2.0 * m * n * k + 4.0 * m * r * (k + n) for _, k, n in parts)
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # A linear's bf16 outputs are 1.7e-3 (2-norm) from their value in 64 bits, its input gradient 2.3e-3.  In a block
    # the codes follow each rounding of the norm's, and of the gate and up, outputs: 9e-3 and 2e-2 there, between
    # two implementations that round at the same points a quarter of it.
    return {"rel": 8e-3, "max": 0.05} if case["kind"] == "linear" else {"rel": 2e-2, "max": 0.2}


# ---------------------------------------------------------------------------------------------------------------
# The same calls in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------------------------
def _hadamard():
    h = torch.ones(1, 1, device=DEV, dtype=torch.float64)
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _rotate(t):
    """Block-diagonal unnormalised Walsh-Hadamard transform of the last axis (its own inverse up to 128)."""
    return (t.reshape(-1, 128) @ _hadamard()).reshape(t.shape)


def _rows_i8(t):
    """Per-row int8 quantization of the rotated rows, rotated back: what the codes stand for."""
    v = _rotate(t)
    s = v.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 127
    return _rotate(torch.round(v / s) * s) / 128


def _base_weight(w, base):
    """The weight that the quantized base stands for, N x K."""
    if base == "fp8":
        amax = w.float().abs().amax(1, keepdim=True).clamp_min(1e-8)
        s = amax / torch.full_like(amax, 448.0)      # a tensor divisor: one correctly rounded division
        q = (w.float() / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return (q.to(torch.bfloat16) * s.to(torch.bfloat16)).double()
    if base == "w8a8":
        return _rows_i8(w.double())
    v = _rotate(w.double()).reshape(w.shape[0], -1, 64)
    s = (v.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 7).to(torch.bfloat16).double()
    return _rotate((torch.round(v / s).clamp(-7, 7) * s).reshape(w.shape)) / 128


class _ExactLinear(torch.autograd.Function):
    """Quantized activations forward, straight through to the input backward."""

    @staticmethod
    def forward(ctx, x, w, a, b, bias, rotated):
        ctx.save_for_backward(x, w, a, b)
        y = (_rows_i8(x) if rotated else x) @ w.t() + (x @ a.t()) @ b.t()
        return y if bias is None else y + bias

    @staticmethod
    def backward(ctx, dy):
        x, w, a, b = ctx.saved_tensors
        g = dy @ b
        return dy @ w + g @ a, None, g.t() @ x, dy.t() @ (x @ a.t()), None, None


def exact(case, seed):
    if case["kind"] == "quantize":
        return None
    if case["kind"] == "linear":
        t = _linear_tensors(case, seed)
        bias = t["bias"]
        if bias is not None:
            bias = (bias.to(torch.bfloat16) if case["base"] == "fp8" else bias).double()
        x = t["x"].double().requires_grad_(case["train"])
        factors = [t["A"].double().requires_grad_(case["train"]), t["B"].double().requires_grad_(case["train"])]
        ys = [_ExactLinear.apply(x, _base_weight(t["w"], case["base"]), *factors, bias, case["base"] != "fp8")]
        dys = [t["dy"]] if case["train"] else None
    else:
        t = _block_tensors(case, seed)
        x = t["x"].double().requires_grad_(case["train"])
        n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (t["norm"].double() + 1)
        h = ((1 + t["scale"].double()) * n + t["shift"].double()).reshape(-1, case["width"])
        factors, by_name = [], {}
        for name, _, _ in _parts(case):
            by_name[name] = [t[p + name].double().requires_grad_(case["train"]) for p in ("A.", "B.")]
            factors += by_name[name]

        def linear(name, v):
            return _ExactLinear.apply(v, _base_weight(t["w." + name], "w8a8"), *by_name[name], None, True)

        if case["kind"] == "attention":
            ys = [linear(name, h) for name, _, _ in _parts(case)]
        else:
            ys = [linear("down", F.silu(linear("gate", h)) * linear("up", h))]
        lead = x.shape[:-1]
        ys = [y.reshape(*lead, y.shape[-1]) for y in ys]
        dys = t["dy"] if case["train"] else None
    if not case["train"]:
        return ys
    grads = torch.autograd.grad(ys, [x, *factors], [d.double() for d in dys])
    return [y.detach() for y in ys] + list(grads)
