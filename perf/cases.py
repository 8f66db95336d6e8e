"""The calls whose speed counts: what a program that trains or runs a Wan or HunyuanVideo model through
this package asks of it, from the text tokens of one denoising step to whole 720P clips.

A case names an operator (``op``), the activation ``[batch, tokens, cols]`` (per-head operators:
``[batch, heads, tokens, cols]`` as the transposed view of the projection's output), whether gradients
are taken (``grad``: forward and backward, as in training; without it the forward alone, as in
sampling) and the parameters' dtype (``params``).  Activations are bfloat16 throughout.  Inputs follow
the distributions of ``teletron_amd.workloads``.
"""
import math

import torch

import teletron_amd
from teletron_amd import reference_api

EPS = 1e-6

# op -> (activations read by forward, written by forward, read by backward, written by backward,
#        parameter vectors per sample [C], row statistics saved for backward)
TRAFFIC = {
    "adaln": (1, 1, 2, 1, 2, 0),
    "rmsnorm": (1, 1, 2, 1, 1, 0),
    "rope": (1, 1, 2, 1, 1, 0),
    "rope_heads": (1, 1, 2, 1, 1, 0),
    "gate": (2, 1, 2, 1, 1, 0),
    "residual_adaln": (2, 2, 3, 1, 2, 0),
    "gated_residual_layernorm": (2, 2, 4, 2, 3, 0),
    "adaln_saved": (1, 2, 2, 1, 2, 1),
}


def _case(op, batch, tokens, cols, *, heads=1, grad=True, params="bfloat16", name=None):
    case = {"op": op, "batch": batch, "tokens": tokens, "cols": cols, "heads": heads, "grad": grad, "params": params}
    return {"name": name, **case} if name else case


def listed():
    return [
        # The smallest call: text-stream AdaLN of a HunyuanVideo double block while sampling, 256 text tokens.
        _case("adaln", 1, 256, 3072, grad=False, name="adaln_text_sampling"),
        # norm_k of Wan-14B's cross attention in training: 512 text tokens.
        _case("rmsnorm", 1, 512, 5120, name="rmsnorm_text_training"),
        # Short clip at Wan-1.3B width through the module form, its weight fp32 as constructed.
        _case("rmsnorm", 2, 4096, 1536, params="float32", name="rmsnorm_small_training"),
        # Ragged width (125 vectors of 8 values), three samples with a modulation of their own each.
        _case("adaln", 3, 5000, 1000, name="adaln_ragged_training"),
        # A width that no vector of 8 values divides.
        _case("rmsnorm", 2, 2500, 1001, name="rmsnorm_odd_training"),
        # Gated residual update of a Wan-1.3B block while sampling with guidance (two samples), 81 frames at 480P.
        _case("gate", 2, 32760, 1536, grad=False, name="gate_480p_sampling"),
        # Wan-1.3B training on four 81-frame 480P clips, per-sample modulation.
        _case("adaln", 4, 32760, 1536, name="adaln_480p_training"),
        # Wan-14B training on an 81-frame 720P clip: the modulated norm in front of attention and MLP.
        _case("adaln", 1, 75600, 5120, name="adaln_720p_training"),
        # The same model's QK-norm with the rotary embedding behind it (40 heads of 128).
        _case("rope", 1, 75600, 5120, heads=40, name="rope_720p_training"),
        # HunyuanVideo's per-head QK-norm with the rotary embedding, 129 frames at 720P, 24 heads.
        _case("rope_heads", 1, 118800, 128, heads=24, name="rope_heads_720p_training"),
        # The largest: Wan-14B's gated attention update and the affine norm that reads it.
        _case("gated_residual_layernorm", 1, 75600, 5120, name="gated_residual_720p_training"),
        # TeleTron's own AdaLN contract (saves x_norm) at the width its kernel has.
        _case("adaln_saved", 1, 118800, 3072, name="adaln_saved_720p_training"),
    ]


def draw(rng):
    """One more case of the same ranges, at most as much traffic as the largest listed one."""
    most = max(work(c)["bytes"] for c in listed())
    while True:
        op = rng.choice(sorted(TRAFFIC))
        grad = rng.random() < 0.7
        batch = rng.choice([1, 1, 2, 3, 4])
        heads, cols = 1, rng.choice([1000, 1536, 2048, 3072, 4096, 5120, 8 * rng.randint(64, 640)])
        tokens = int(256 * math.exp(rng.random() * math.log(118800 / 256)))
        params = "bfloat16"
        if op == "rmsnorm":
            params = rng.choice(["bfloat16", "float32"])
        if op in ("rmsnorm", "adaln") and rng.random() < 0.25:
            cols, tokens = rng.randint(500, 2100), min(tokens, 8192)      # any width at all
        if op == "rope":
            heads = rng.choice([12, 16, 24, 40])
            cols = heads * 128
        if op == "rope_heads":
            heads, cols = rng.choice([12, 16, 24, 24, 40]), rng.choice([64, 128])
        if op == "adaln_saved":
            batch, cols = 1, rng.choice([1536, 3072, 3072, 5120])
        case = _case(op, batch, tokens, cols, heads=heads, grad=grad, params=params)
        if work(case)["bytes"] <= most:
            return case


def _randn(shape, g, mean=0.0, std=1.0, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device=g.device, dtype=torch.float32).mul_(std).add_(mean).to(dtype)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, b, s, c, h = (case[k] for k in ("op", "batch", "tokens", "cols", "heads"))
    dtype = getattr(torch, case["params"])
    state = {"case": case, "call": None, "inputs": [], "grads": []}

    def activation():
        if op == "rope_heads":        # [B, H, S, D], the transposed view of the projection's [B, S, H * D]
            return _randn((b, s, h, c), g).transpose(1, 2)
        return _randn((b, s, c), g)

    x = activation()
    if op in ("adaln", "adaln_saved", "residual_adaln"):
        shift, scale = _randn((b, 6, c), g, std=0.1, dtype=dtype).chunk(6, dim=1)[:2]     # as a DiT block cuts its modulation
    if op == "adaln":
        norm = teletron_amd.FusedAdaLN(c, eps=EPS)
        state["call"], state["inputs"] = norm, [x, shift, scale]
    elif op == "adaln_saved":
        shift, scale = shift.reshape(c), scale.reshape(c)
        state["call"] = lambda x, scale, shift: reference_api.AdaLNModelFunction.apply(x, scale, shift, EPS, c)
        state["inputs"] = [x, scale, shift]
    elif op == "rmsnorm":
        norm = teletron_amd.FusedRMSNorm(c, eps=EPS).to(device="cuda", dtype=dtype)
        with torch.no_grad():
            norm.weight.copy_(_randn((c,), g, mean=1.0, std=0.1, dtype=dtype))
        state["call"], state["inputs"] = (lambda x, weight: norm(x)), [x, norm.weight]
    elif op in ("rope", "rope_heads"):
        weight = _randn((c,), g, mean=1.0, std=0.1, dtype=dtype)
        d = c // h if op == "rope" else c
        angles = _randn((s, d // 2), g, std=3.0, dtype=torch.float32)
        table = torch.stack([angles.cos(), angles.sin()], dim=-1)       # built once per step, shared by all blocks
        state["table"] = table
        if op == "rope":
            state["call"] = lambda x, weight: teletron_amd.RMSNormRopeFunction.apply(x, weight, table, EPS, h)
        else:
            state["call"] = lambda x, weight: teletron_amd.RMSNormRopeHeadsFunction.apply(x, weight, table, EPS)
        state["inputs"] = [x, weight]
    elif op == "gate":
        gate = _randn((b, 6, c), g, std=0.5, dtype=dtype).chunk(6, dim=1)[2]
        state["call"], state["inputs"] = teletron_amd.FusedGate(), [x, gate, activation()]
    elif op == "residual_adaln":
        state["call"] = lambda x, r, shift, scale: teletron_amd.residual_adaln(x, r, None, shift, scale, EPS)
        state["inputs"] = [x, activation(), shift, scale]
    elif op == "gated_residual_layernorm":
        gate = _randn((b, 6, c), g, std=0.5, dtype=dtype).chunk(6, dim=1)[2]
        weight = _randn((c,), g, mean=1.0, std=0.1, dtype=dtype)
        bias = _randn((c,), g, std=0.1, dtype=dtype)
        state["call"] = lambda x, r, gate, weight, bias: teletron_amd.residual_layer_norm(x, r, gate, weight, bias, EPS)
        state["inputs"] = [x, activation(), gate, weight, bias]
    else:
        raise ValueError(op)
    if case["grad"]:
        state["inputs"] = [t if t.requires_grad else t.detach().requires_grad_(True) for t in state["inputs"]]
        state["grads"] = [activation() for _ in range(2 if "residual_" in op else 1)]
    return state


def run(state):
    if not state["case"]["grad"]:
        with torch.no_grad():
            return state["call"](*state["inputs"])
    out = state["call"](*state["inputs"])
    outs = list(out) if isinstance(out, tuple) else [out]
    return outs + list(torch.autograd.grad(outs, state["inputs"], state["grads"]))


def exact(case, seed):
    """What ``run`` returns, by the formulas in 64 bits (gradients by autograd)."""
    state = prepare(case, seed)
    op, c, h = case["op"], case["cols"], case["heads"]
    inputs = [t.detach().double().requires_grad_(case["grad"]) for t in state["inputs"]]

    def layer_norm(v):
        d = v - v.mean(dim=-1, keepdim=True)
        return d * torch.rsqrt(d.square().mean(dim=-1, keepdim=True) + EPS)

    def rms_norm(v, weight):
        return v * torch.rsqrt(v.square().mean(dim=-1, keepdim=True) + EPS) * weight

    def rotate(v):                  # [..., tokens, D], pairs of neighbouring values
        cos, sin = state["table"].double().unbind(-1)
        re, im = v[..., 0::2], v[..., 1::2]
        return torch.stack([re * cos - im * sin, re * sin + im * cos], dim=-1).flatten(-2)

    if op == "adaln":
        x, shift, scale = inputs
        outs = [layer_norm(x) * (1 + scale) + shift]
    elif op == "adaln_saved":
        x, scale, shift = inputs
        outs = [layer_norm(x) * (1 + scale) + shift]
    elif op == "rmsnorm":
        outs = [rms_norm(*inputs)]
    elif op == "rope":
        outs = [rotate(rms_norm(*inputs).unflatten(-1, (h, c // h)).transpose(1, 2)).transpose(1, 2).flatten(-2)]
    elif op == "rope_heads":
        outs = [rotate(rms_norm(*inputs))]
    elif op == "gate":
        x, gate, residual = inputs
        outs = [x + gate * residual]
    elif op == "residual_adaln":
        x, residual, shift, scale = inputs
        s = x + residual
        outs = [s, layer_norm(s) * (1 + scale) + shift]
    else:
        x, residual, gate, weight, bias = inputs
        s = x + gate * residual
        outs = [s, layer_norm(s) * weight + bias]
    if not case["grad"]:
        return outs[0] if len(outs) == 1 else tuple(outs)
    grads = torch.autograd.grad(outs, inputs, [g.double() for g in state["grads"]])
    return [o.detach() for o in outs] + list(grads)


def work(case):
    """Every activation, parameter, table and gradient once; the arithmetic is a few operations a value."""
    op, b, s, c, h = (case[k] for k in ("op", "batch", "tokens", "cols", "heads"))
    elements = b * s * c * (h if op == "rope_heads" else 1)
    read_f, written_f, read_b, written_b, vectors, stats = TRAFFIC[op]
    per_sample = b if op in ("adaln", "residual_adaln", "gate") else 1
    params = vectors * per_sample * c * (4 if case["params"] == "float32" else 2)
    table = 4 * s * (c // h if op == "rope" else c) if op in ("rope", "rope_heads") else 0
    rows = stats * b * s * 4
    total = 2 * elements * (read_f + written_f) + params + table + rows
    flops = 8 * elements
    if case["grad"]:
        total += 2 * elements * (read_b + written_b) + 2 * params + table + rows
        flops += 16 * elements
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """bfloat16 results: one rounding of values computed in fp32.  Against the same formulas in 64 bits most
    outputs are off by 1.7e-3 (2-norm) and by half a bfloat16 step (3.9e-3) at the worst value; the worst
    are 2.5e-3 and 8.8e-3, where a value rounded before enters (an fp32 weight, the updated residual
    stream, the saved x_norm).  Stated four times as large."""
    return {"rel": 1e-2, "max": 3.5e-2}
