"""The calls a user of this package makes, as cases to be timed and compared.

A case is a dict of plain values; ``kind`` names the entry point:

* ``scan``       ``suffix_scan_pullbacks`` (``cotangents`` false) or ``suffix_scan_pullbacks_and_cotangents``
* ``chain``      ``suffix_scan_cotangents``: the cotangents without the matrices
* ``attention``  ``attention_input_pullback_basis``: dQ, dK, dV for ``P`` directions
* ``region``     ``HipTransformerLowering.input_pullback_basis``: a range of Transformer layers, ``P`` directions
* ``vjp``        ``HipTransformerLowering.parameter_vjp``: the parameter gradients of such a range, one cotangent

``listed()`` holds the cases of the benchmark and of the reference's own programs, ``draw`` more of the same ranges.
Everything ``prepare`` makes comes from a generator on the GPU with the given seed.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

from latent_bounded_interfaces_amd.backends import HipTransformerLowering
from latent_bounded_interfaces_amd.hip.interface import (suffix_scan_cotangents, suffix_scan_pullbacks,
                                                         suffix_scan_pullbacks_and_cotangents)
from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
_CONV_TAPS = 4   # depthwise causal convolution on the packed projection, the blocks' default
_ROPE_BASE = 10000.0
_NORM_EPS = 1e-5

# what one call may cost: the largest listed ones, and for fp32 / non-causal attention the small models and gradient
# checks that such calls come from
_ATTENTION_FLOPS = 9e12
_ATTENTION_CHECK_FLOPS = 6e10
_REGION_FLOPS = 1.6e13
_REGION_FP32_FLOPS = 3e11


def listed():
    return [
        # The smallest scan of the benchmark, which the reference's own CPU path runs too: latency and launches.
        {"name": "scan_small", "kind": "scan", "B": 4, "K": 8, "d": 32, "dtype": "fp32", "cotangents": True},
        # One sequence through a deep stack of wide interfaces: the batch of the reference's tests and launchers.
        {"name": "scan_single", "kind": "scan", "B": 1, "K": 128, "d": 256, "dtype": "fp32", "cotangents": True},
        # The benchmark's headline: a training batch, every suffix matrix and every cotangent.
        {"name": "scan_full", "kind": "scan", "B": 64, "K": 128, "d": 256, "dtype": "fp32", "cotangents": True},
        # The same from 16-bit storage.
        {"name": "scan_bf16", "kind": "scan", "B": 64, "K": 128, "d": 256, "dtype": "bf16", "cotangents": True},
        # An interface width that is no power of two, suffix matrices only (Jacobian diagnostics).
        {"name": "scan_ragged", "kind": "scan", "B": 16, "K": 50, "d": 96, "dtype": "fp32", "cotangents": False},
        # The reference's own attention benchmark shape: one short launch.
        {"name": "attention_small", "kind": "attention", "B": 8, "H": 8, "T": 128, "Dh": 64, "P": 4, "dtype": "fp16",
         "causal": True},
        # Long context, wide heads, many directions: the largest attention call.
        {"name": "attention_long", "kind": "attention", "B": 4, "H": 16, "T": 4096, "Dh": 128, "P": 16,
         "dtype": "bf16", "causal": True},
        # A sequence length that is no multiple of any tile.
        {"name": "attention_ragged", "kind": "attention", "B": 8, "H": 12, "T": 1000, "Dh": 64, "P": 16,
         "dtype": "bf16", "causal": True},
        # Full precision: gradient checks and models trained without autocast.
        {"name": "attention_fp32", "kind": "attention", "B": 4, "H": 8, "T": 512, "Dh": 64, "P": 8, "dtype": "fp32",
         "causal": True},
        # One region of a small model, short sequence, grouped keys, a general basis: many small launches.
        {"name": "region_small", "kind": "region", "layers": 2, "dim": 256, "heads": 4, "kv_heads": 2, "head_dim": 64,
         "B": 1, "T": 128, "P": 16, "dtype": "bf16", "constant": False},
        # One region of the end-to-end configuration; the mean-pooling interface of width 64 sends 64 directions
        # back, each the same at every position.
        {"name": "region_full", "kind": "region", "layers": 2, "dim": 768, "heads": 12, "kv_heads": 12, "head_dim": 64,
         "B": 8, "T": 1024, "P": 64, "dtype": "bf16", "constant": True},
        # The parameter gradients of that region: the other half of a training step.
        {"name": "vjp_full", "kind": "vjp", "layers": 2, "dim": 768, "heads": 12, "kv_heads": 12, "head_dim": 64,
         "B": 8, "T": 1024, "dtype": "bf16"},
    ]


def _spread(rng, low, high):
    """A whole number, spread over the logarithm of its range."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_scan(rng, kind):
    case = {"kind": kind, "B": _spread(rng, 1, 64), "K": _spread(rng, 4, 128),
            "d": rng.choice([32, 64, 128, 256, _spread(rng, 12, 256), _spread(rng, 12, 256)]),
            "dtype": rng.choice(["fp32", "fp32", "bf16", "fp16"])}
    if kind == "scan":
        case["cotangents"] = rng.random() < 0.6
    return case


def _draw_attention(rng):
    while True:
        case = {"kind": "attention", "B": _spread(rng, 1, 8), "H": _spread(rng, 1, 16),
                "T": rng.choice([64 * _spread(rng, 1, 64), _spread(rng, 24, 4096)]),
                "Dh": rng.choice([64, 64, 128, 128, 32, 80, 96]), "P": _spread(rng, 1, 16),
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "causal": rng.random() < 0.85}
        plain = case["dtype"] != "fp32" and case["causal"]
        if 1e7 <= work(case)["flops"] <= (_ATTENTION_FLOPS if plain else _ATTENTION_CHECK_FLOPS):
            return case


def _draw_region(rng, kind):
    while True:
        heads, head_dim = rng.choice([(4, 64), (8, 64), (12, 64), (4, 128), (8, 32)])
        case = {"kind": kind, "layers": rng.choice([1, 2]), "dim": heads * head_dim, "heads": heads,
                "kv_heads": rng.choice([heads, heads, heads // 2]), "head_dim": head_dim, "B": _spread(rng, 1, 8),
                "T": rng.choice([64 * _spread(rng, 1, 16), _spread(rng, 48, 1024)]),
                "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])}
        if kind == "region":
            case["P"], case["constant"] = _spread(rng, 4, 64), rng.random() < 0.6
        if work(case)["flops"] <= (_REGION_FP32_FLOPS if case["dtype"] == "fp32" else _REGION_FLOPS):
            return case


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "chain", "attention", "attention", "attention", "region", "region", "vjp"])
    if kind in ("scan", "chain"):
        return _draw_scan(rng, kind)
    if kind == "attention":
        return _draw_attention(rng)
    return _draw_region(rng, kind)


# ---------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------
class _Node(torch.nn.Module):
    """A holder of parameters and plain attributes, named as the reference's modules are."""


class _Source:
    """Normal values on the GPU from one seeded generator."""

    def __init__(self, seed):
        self.device = torch.device("cuda")
        self.gen = torch.Generator(device=self.device).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return torch.randn(shape, generator=self.gen, device=self.device).mul_(std).to(dtype)


def _interface_matrices(src, case):
    """State Jacobians of a residual interface: the identity and a small update."""
    width = case["d"]
    mats = src.normal(case["B"], case["K"], width, width, std=(0.01 / width) ** 0.5)
    mats.diagonal(dim1=-2, dim2=-1).add_(1.0)
    return mats.to(_DTYPES[case["dtype"]])


def _rms_norm(x, norm):
    x = x.to(norm.weight.dtype)
    wide = x.float()
    return (wide * torch.rsqrt(wide.pow(2).mean(-1, keepdim=True) + norm.eps)).to(x.dtype) * norm.weight


def _rotated(x):
    half = x.shape[-1] // 2
    position = torch.arange(x.shape[-2], device=x.device, dtype=torch.float32)
    freq = _ROPE_BASE ** (-torch.arange(half, device=x.device, dtype=torch.float32) / half)
    angle = torch.outer(position, freq)
    a, b = x[..., :half].float(), x[..., half:].float()
    return torch.cat((a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()), dim=-1).to(x.dtype)


def _make_block(src, case, dtype):
    dim, heads, kv_heads, head_dim = case["dim"], case["heads"], case["kv_heads"], case["head_dim"]
    hidden, packed = 4 * dim, (heads + 2 * kv_heads) * head_dim

    def weight(*shape, std):
        return torch.nn.Parameter(src.normal(*shape, std=std, dtype=dtype))

    def linear(out_features, in_features):
        node = _Node()
        node.weight, node.bias = weight(out_features, in_features, std=in_features ** -0.5), None
        return node

    def norm():
        node = _Node()
        node.weight = torch.nn.Parameter((1.0 + src.normal(dim, std=0.1)).to(dtype))
        node.eps = _NORM_EPS
        return node

    attn, mlp, block = _Node(), _Node(), _Node()
    attn.n_heads, attn.n_kv_heads, attn.head_dim, attn.d_conv = heads, kv_heads, head_dim, _CONV_TAPS
    attn.rope_base, attn.rope_interleaved, attn.softmax_scale = _ROPE_BASE, False, None
    attn.in_proj, attn.out_proj = linear(packed, dim), linear(dim, heads * head_dim)
    attn.conv1d = _Node()
    attn.conv1d.weight, attn.conv1d.bias = weight(packed, 1, _CONV_TAPS, std=_CONV_TAPS ** -0.5), None
    mlp.fc1, mlp.fc2 = linear(2 * hidden, dim), linear(dim, hidden)
    block.norm, block.norm2, block.attn, block.mlp, block.residual_in_fp32 = norm(), norm(), attn, mlp, True
    return block


def _forward_block(block, hidden, residual):
    """The block as the model's forward runs it, with the cache that it leaves behind."""
    attn, mlp = block.attn, block.mlp
    batch, seq_len, _ = hidden.shape
    norm1_input = hidden if residual is None else hidden + residual
    residual = norm1_input.float()
    normed1 = _rms_norm(norm1_input, block.norm)
    packed = F.linear(normed1, attn.in_proj.weight)
    shifted = F.pad(packed, (0, 0, _CONV_TAPS - 1, 0))
    packed = sum(shifted[:, j:j + seq_len] * attn.conv1d.weight[:, 0, j] for j in range(_CONV_TAPS))
    q_width, kv_width = attn.n_heads * attn.head_dim, attn.n_kv_heads * attn.head_dim
    q, k, v = (t.reshape(batch, seq_len, -1, attn.head_dim).transpose(1, 2)
               for t in packed.split((q_width, kv_width, kv_width), dim=-1))
    repeats = attn.n_heads // attn.n_kv_heads
    q, k, v = _rotated(q), _rotated(k).repeat_interleave(repeats, dim=1), v.repeat_interleave(repeats, dim=1)
    heads = F.scaled_dot_product_attention(q, k, v, is_causal=True)
    merged = heads.transpose(1, 2).reshape(batch, seq_len, q_width)
    norm2_input = F.linear(merged, attn.out_proj.weight) + residual
    normed2 = _rms_norm(norm2_input, block.norm2)
    fc1 = F.linear(normed2, mlp.fc1.weight)
    up, gate = fc1.chunk(2, dim=-1)
    down_input = up * F.silu(gate)
    hidden = F.linear(down_input, mlp.fc2.weight)
    cache = SimpleNamespace(
        attention=SimpleNamespace(norm_input=norm1_input, norm_output=normed1, q_rope=q, k_expanded=k, v_expanded=v,
                                  out_proj_input=merged),
        mlp=SimpleNamespace(norm_input=norm2_input, norm_output=normed2, fc1_output=fc1, down_input=down_input))
    return hidden, norm2_input, cache


@torch.no_grad()
def _make_region(src, case):
    """A region of a model at initialisation, and the forward cache of one batch through it."""
    dtype = _DTYPES[case["dtype"]]
    backend = _Node()
    backend.backbone = _Node()
    backend.backbone.blocks = torch.nn.ModuleList(_make_block(src, case, dtype) for _ in range(case["layers"]))
    region_input = src.normal(case["B"], case["T"], case["dim"], dtype=dtype)
    hidden, residual, caches = region_input, None, []
    for index, block in enumerate(backend.backbone.blocks):
        hidden, residual, cache = _forward_block(block, hidden, residual)
        cache.layer_index = index
        caches.append(cache)
    return backend, SimpleNamespace(region_index=0, layer_range=(0, case["layers"]), layer_caches=caches,
                                    region_input=region_input)


def prepare(case, seed):
    src, kind = _Source(seed), case["kind"]
    state = SimpleNamespace(kind=kind)
    if kind in ("scan", "chain"):
        state.mats = _interface_matrices(src, case)
        state.g = src.normal(case["B"], case["d"]) if case.get("cotangents", True) else None
    elif kind == "attention":
        shape, dtype = (case["H"], case["T"], case["Dh"]), _DTYPES[case["dtype"]]
        state.qkv = [src.normal(case["B"], *shape, dtype=dtype) for _ in range(3)]
        state.d_out = src.normal(case["B"], case["P"], *shape, dtype=dtype)
        state.scale, state.causal = 1.0 / math.sqrt(case["Dh"]), case["causal"]
    else:
        state.lowering = HipTransformerLowering()
        state.backend, state.cache = _make_region(src, case)
        if kind == "vjp":
            state.cotangent = src.normal(case["B"], case["T"], case["dim"])
        elif case["constant"]:  # mean pooling: one cotangent per direction, 1/T of it at every position
            pooled = src.normal(case["B"], case["P"], 1, case["dim"], std=1.0 / case["T"])
            state.basis = pooled.expand(-1, -1, case["T"], -1)
        else:
            state.basis = src.normal(case["B"], case["P"], case["T"], case["dim"])
    return state


# ---------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------
def run(state):
    if state.kind == "scan":
        if state.g is None:
            return suffix_scan_pullbacks(state.mats)
        return suffix_scan_pullbacks_and_cotangents(state.mats, state.g)
    if state.kind == "chain":
        return suffix_scan_cotangents(state.mats, state.g)
    if state.kind == "attention":
        return attention_input_pullback_basis(*state.qkv, state.d_out, softmax_scale=state.scale, causal=state.causal,
                                              kernel_mode="hip")
    if state.kind == "region":
        return state.lowering.input_pullback_basis(backend=state.backend, cache=state.cache,
                                                   output_cotangent_basis=state.basis)
    return state.lowering.parameter_vjp(backend=state.backend, cache=state.cache, output_cotangent=state.cotangent)


# ---------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------
def _attention_flops(batch, heads, seq_len, head_dim, basis, causal):
    """Q K^T once, then dP, dV, dQ, dK for every direction."""
    pairs = seq_len * (seq_len + 1) / 2 if causal else seq_len * seq_len
    return batch * heads * pairs * 2.0 * head_dim * (1 + 4 * basis)


def _region_work(case):
    size, layers, basis = _BYTES[case["dtype"]], case["layers"], case.get("P", 1)
    dim, hidden, q_width = case["dim"], 4 * case["dim"], case["heads"] * case["head_dim"]
    packed = q_width + 2 * case["kv_heads"] * case["head_dim"]
    positions = case["B"] * case["T"]
    rows = positions * basis
    weights = packed * dim + dim * q_width + 3 * hidden * dim
    attention = _attention_flops(case["B"], case["heads"], case["T"], case["head_dim"], basis, True)
    # per position and layer: two norm inputs (fp32 but for the first), q, k, v, the gated MLP's 2 hidden inputs
    cache = positions * (8 * dim + size * (3 * q_width + 2 * hidden)) * layers - positions * (4 - size) * dim
    flops = layers * (2.0 * rows * weights + attention)
    nbytes = cache + size * layers * (weights + packed * _CONV_TAPS + 2 * dim)
    if case["kind"] == "vjp":
        # a second product per weight, the projection in front of the convolution once more; module inputs, gradients
        flops += layers * 2.0 * positions * (weights + packed * dim)
        nbytes += size * layers * (positions * (2 * dim + q_width + hidden) + weights + packed * _CONV_TAPS + 2 * dim)
        nbytes += 4 * positions * dim
    else:
        if case["constant"]:  # the last down projection sees one row per direction
            flops -= 2.0 * (rows - case["B"] * basis) * hidden * dim
        nbytes += 4 * dim * (rows + (case["B"] * basis if case["constant"] else rows))
    return {"bytes": float(nbytes), "flops": flops}


def work(case):
    kind, size = case["kind"], _BYTES[case["dtype"]]
    if kind in ("scan", "chain"):
        matrices, width = case["B"] * case["K"], case["d"]
        nbytes, flops = float(matrices * width * width * size), 0.0
        if kind == "scan":
            nbytes += 4.0 * case["B"] * (case["K"] + 1) * width * width
            flops += case["B"] * (case["K"] - 1) * 2.0 * width ** 3
        if case.get("cotangents", True):
            nbytes += 4.0 * case["B"] * (case["K"] + 2) * width
            flops += 2.0 * matrices * width * width
        return {"bytes": nbytes, "flops": flops}
    if kind == "attention":
        values = case["B"] * case["H"] * case["T"] * case["Dh"]
        return {"bytes": float(values * size * (3 + 4 * case["P"])),
                "flops": _attention_flops(case["B"], case["H"], case["T"], case["Dh"], case["P"], case["causal"])}
    return _region_work(case)


def tolerance(case):
    """About four times the relative error against a 64-bit evaluation of the same inputs (16-bit regions: against the
    fp32 path on the same rounded weights and activations)."""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "chain" or (kind == "scan" and dtype != "bf16"):
        return {"rel": 8e-6}   # 1.1e-6 in the matrices and 1.8e-6 in the cotangents at K = 128, d = 256
    if kind == "scan":
        return {"rel": 1e-4}   # 2.2e-5: the running product in 16 significand bits
    if kind == "attention":
        return {"rel": {"fp32": 3e-6, "fp16": 1.5e-3, "bf16": 1.2e-2}[dtype]}   # 6e-7, 3.7e-4, 3.0e-3
    if kind == "region":
        return {"rel": {"fp32": 5e-6, "fp16": 2e-3, "bf16": 1.5e-2}[dtype]}     # 0.9e-6, 4.5e-4, 3.9e-3
    return {"rel": {"fp32": 6e-6, "fp16": 3.5e-3, "bf16": 2.5e-2}[dtype]}       # 1.4e-6, 8.4e-4, 6.8e-3
