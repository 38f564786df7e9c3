"""Region-level input pullback of a Transformer layer range for P cotangent directions.

Implements ``TransformerLowering.input_pullback_basis`` of the reference
(backends/transformer.py:64-75; the CUDA class leaves it as a stub,
backends/transformer_cuda.py:45-64) for the block the reference's backend executes
(backends/transformer.py:118-246):

    res1 = hidden (+ residual);  a = out_proj(attention(rope(split(conv1d(in_proj(norm(res1)))))))
    res2 = a + res1;             m = fc2(up * silu(gate)),  [up | gate] = fc1(norm2(res2))
    region_output = m + res2 of the last layer

The cotangent basis [B, P, T, D] is pulled back through the layers in reverse.  Matrix
products are library GEMMs on the [B*P*T, *] cotangent rows (small ones
``lbi_small_product``, weight gradients ``lbi_weight_gradient``); everything between them
runs in the kernels of liblbi_hip.so (RMSNorm, gated MLP, head split, rotary embedding + KV-group
sum, causal convolution, and the attention pullback itself).  The residual-stream cotangent
is kept in fp32, branch cotangents in the dtype of the weights.  Inputs are read from the
forward cache the backend recorded; nothing is recomputed except the softmax statistics
inside the attention kernel.  GPU only.
"""
from __future__ import annotations

import ctypes
import math
from typing import Any

import torch

from ... import _lib
from . import _MFMA_HEAD_DIMS, _MFMA_SEQ_MULTIPLE, _SINGLE_LAUNCH_MAX_SEQ, attention_input_pullback_basis


def _stream(t: torch.Tensor) -> int:
    return _lib.current_stream_ptr(t.device)


def _require_cuda(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if not t.is_cuda:
            raise RuntimeError("region pullback tensors must be CUDA tensors (this build has no CPU execution path)")


def rmsnorm_pullback(g_out: torch.Tensor, x: torch.Tensor, weight: torch.Tensor, eps: float,
                     g_residual: torch.Tensor | None, *, want_branch: bool,
                     keep_residual: bool = False) -> tuple[torch.Tensor, torch.Tensor | None]:
    """``g_out [B,P,T,D]`` through RMSNorm at input ``x [B,T,D]``, plus ``g_residual`` (fp32).

    Returns ``(sum fp32, sum in g_out.dtype or None)``.  ``g_residual [B,P,T,D]`` is overwritten with the
    sum unless ``keep_residual``; ``g_residual [B,P,1,D]`` (the same cotangent at every position) is read only.
    """
    _require_cuda(g_out, x, weight)
    bsz, basis, seqlen, dim = g_out.shape
    if x.shape != (bsz, seqlen, dim) or weight.shape != (dim,):
        raise ValueError("rmsnorm_pullback: x must be [B, T, D] and weight [D] matching g_out [B, P, T, D]")
    g_out, x, weight = g_out.contiguous(), x.contiguous(), weight.to(g_out.dtype).contiguous()
    shared = 0
    if g_residual is None:
        total = torch.empty(g_out.shape, device=g_out.device, dtype=torch.float32)
        res_ptr = None
    else:
        if g_residual.dtype != torch.float32 or not g_residual.is_contiguous():
            raise ValueError("rmsnorm_pullback: g_residual must be a contiguous fp32 tensor")
        if g_residual.shape == g_out.shape:
            total = torch.empty_like(g_residual) if keep_residual else g_residual
        elif g_residual.shape == (bsz, basis, 1, dim):
            total = torch.empty(g_out.shape, device=g_out.device, dtype=torch.float32)
            shared = 1
        else:
            raise ValueError("rmsnorm_pullback: g_residual must be shaped like g_out, or [B, P, 1, D]")
        res_ptr = g_residual.data_ptr()
    branch = torch.empty_like(g_out) if want_branch else None
    with _lib.device_guard(g_out.device):
        status = _lib.load().lbi_rmsnorm_pullback(
            g_out.data_ptr(), x.data_ptr(), weight.data_ptr(), res_ptr, total.data_ptr(),
            branch.data_ptr() if branch is not None else None, bsz, basis, seqlen, dim, float(eps), shared,
            _lib.dtype_code(g_out.dtype), _lib.dtype_code(x.dtype), _stream(g_out))
    _lib.check(status, "lbi_rmsnorm_pullback")
    return total, branch


def gated_mlp_pullback(g_down_input: torch.Tensor, fc1_output: torch.Tensor) -> torch.Tensor:
    """``g_down_input [B,P,T,Hd]`` (or ``[B,P,1,Hd]``: the same at every position), ``fc1_output [B,T,2Hd]``
    -> cotangent of fc1_output ``[B,P,T,2Hd]``."""
    _require_cuda(g_down_input, fc1_output)
    bsz, basis, g_len, hidden = g_down_input.shape
    if fc1_output.dim() != 3 or fc1_output.shape[0] != bsz or fc1_output.shape[2] != 2 * hidden \
            or fc1_output.dtype != g_down_input.dtype:
        raise ValueError("gated_mlp_pullback: fc1_output must be [B, T, 2*hidden] in the dtype of g_down_input")
    seqlen = int(fc1_output.shape[1])
    if g_len != seqlen and g_len != 1:
        raise ValueError("gated_mlp_pullback: g_down_input must be [B, P, T, hidden] or [B, P, 1, hidden]")
    shared = int(g_len == 1 and seqlen != 1)
    g_down_input, fc1_output = g_down_input.contiguous(), fc1_output.contiguous()
    out = torch.empty((bsz, basis, seqlen, 2 * hidden), device=g_down_input.device, dtype=g_down_input.dtype)
    with _lib.device_guard(out.device):
        status = _lib.load().lbi_gated_mlp_pullback(
            g_down_input.data_ptr(), fc1_output.data_ptr(), out.data_ptr(), bsz, basis, seqlen, hidden, shared,
            _lib.dtype_code(out.dtype), _stream(out))
    _lib.check(status, "lbi_gated_mlp_pullback")
    return out


def attn_heads_split(g_merged: torch.Tensor, n_heads: int, head_dim: int) -> torch.Tensor:
    """``[B,P,T,H*Dh]`` -> ``[B,P,H,T,Dh]``."""
    _require_cuda(g_merged)
    bsz, basis, seqlen, width = g_merged.shape
    if width != n_heads * head_dim:
        raise ValueError("attn_heads_split: last dimension must be n_heads * head_dim")
    g_merged = g_merged.contiguous()
    out = torch.empty((bsz, basis, n_heads, seqlen, head_dim), device=g_merged.device, dtype=g_merged.dtype)
    with _lib.device_guard(out.device):
        status = _lib.load().lbi_attn_heads_split(g_merged.data_ptr(), out.data_ptr(), bsz, basis, seqlen, n_heads,
                                                  head_dim, _lib.dtype_code(out.dtype), _stream(out))
    _lib.check(status, "lbi_attn_heads_split")
    return out


_ROPE_TABLES: dict[tuple, tuple[torch.Tensor, torch.Tensor]] = {}


def rope_tables(seq_len: int, head_dim: int, base: float, device: torch.device) -> tuple[torch.Tensor, torch.Tensor]:
    """cos, sin ``[T, Dh/2]`` fp32 of the rotary angles, built as the reference's apply_rope does
    (backbones/transformer/rope.py:14-20) and cached per (T, Dh, base, device)."""
    key = (seq_len, head_dim, float(base), str(device))
    hit = _ROPE_TABLES.get(key)
    if hit is None:
        half = head_dim // 2
        positions = torch.arange(seq_len, device=device, dtype=torch.float32)
        freq_seq = torch.arange(half, device=device, dtype=torch.float32)
        freqs = torch.outer(positions, base ** (-2.0 * freq_seq / float(head_dim)))
        hit = (freqs.cos().contiguous(), freqs.sin().contiguous())
        if len(_ROPE_TABLES) > 32:
            _ROPE_TABLES.clear()
        _ROPE_TABLES[key] = hit
    return hit


def attn_qkv_pullback(dq: torch.Tensor, dk: torch.Tensor, dv: torch.Tensor, *, n_kv_heads: int, rope_base: float,
                      rope_interleaved: bool) -> torch.Tensor:
    """``dq, dk, dv [B,P,H,T,Dh]`` -> cotangent of the packed projection ``[B,P,T,(H+2Hkv)*Dh]``."""
    _require_cuda(dq, dk, dv)
    bsz, basis, heads, seqlen, head_dim = dq.shape
    if dk.shape != dq.shape or dv.shape != dq.shape or dk.dtype != dq.dtype or dv.dtype != dq.dtype:
        raise ValueError("attn_qkv_pullback: dq, dk, dv must share shape [B, P, H, T, Dh] and dtype")
    if heads % n_kv_heads:
        raise ValueError("n_heads must be divisible by n_kv_heads")
    if head_dim % 2:
        raise ValueError("RoPE requires an even head dimension.")
    dq, dk, dv = dq.contiguous(), dk.contiguous(), dv.contiguous()
    cos, sin = rope_tables(seqlen, head_dim, rope_base, dq.device)
    out = torch.empty((bsz, basis, seqlen, (heads + 2 * n_kv_heads) * head_dim), device=dq.device, dtype=dq.dtype)
    with _lib.device_guard(out.device):
        status = _lib.load().lbi_attn_qkv_pullback(
            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), cos.data_ptr(), sin.data_ptr(), out.data_ptr(), bsz, basis,
            seqlen, heads, n_kv_heads, head_dim, int(bool(rope_interleaved)), _lib.dtype_code(out.dtype), _stream(out))
    _lib.check(status, "lbi_attn_qkv_pullback")
    return out


def causal_conv1d_pullback(g_out: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``g_out [B,P,T,C]`` through the depthwise causal convolution with ``weight [C,1,k]``."""
    _require_cuda(g_out, weight)
    bsz, basis, seqlen, channels = g_out.shape
    if weight.dim() != 3 or weight.shape[0] != channels or weight.shape[1] != 1:
        raise ValueError("causal_conv1d_pullback: weight must be [C, 1, k] (depthwise)")
    g_out = g_out.contiguous()
    weight = weight.to(g_out.dtype).contiguous()
    out = torch.empty_like(g_out)
    with _lib.device_guard(out.device):
        status = _lib.load().lbi_causal_conv1d_pullback(g_out.data_ptr(), weight.data_ptr(), out.data_ptr(),
                                                        bsz * basis, seqlen, channels, weight.shape[-1],
                                                        _lib.dtype_code(out.dtype), _stream(out))
    _lib.check(status, "lbi_causal_conv1d_pullback")
    return out


#: longest convolution filter the one-pass projection + convolution pullback takes
FUSED_CONV_MAX_TAPS = 8


def attn_qkv_conv_pullback(dq: torch.Tensor, dk: torch.Tensor, dv: torch.Tensor, conv_weight: torch.Tensor, *,
                           n_kv_heads: int, rope_base: float, rope_interleaved: bool) -> torch.Tensor:
    """:func:`attn_qkv_pullback` then :func:`causal_conv1d_pullback` in one pass over ``dq, dk, dv``
    (same arithmetic as the two calls, bit-identical in fp32; filters of at most ``FUSED_CONV_MAX_TAPS`` taps)."""
    _require_cuda(dq, dk, dv, conv_weight)
    bsz, basis, heads, seqlen, head_dim = dq.shape
    if dk.shape != dq.shape or dv.shape != dq.shape or dk.dtype != dq.dtype or dv.dtype != dq.dtype:
        raise ValueError("attn_qkv_conv_pullback: dq, dk, dv must share shape [B, P, H, T, Dh] and dtype")
    if heads % n_kv_heads:
        raise ValueError("n_heads must be divisible by n_kv_heads")
    if head_dim % 2:
        raise ValueError("RoPE requires an even head dimension.")
    channels = (heads + 2 * n_kv_heads) * head_dim
    if conv_weight.dim() != 3 or conv_weight.shape[0] != channels or conv_weight.shape[1] != 1:
        raise ValueError("attn_qkv_conv_pullback: weight must be [C, 1, k] (depthwise) with C = (H + 2 Hkv) Dh")
    dq, dk, dv = dq.contiguous(), dk.contiguous(), dv.contiguous()
    weight = conv_weight.to(dq.dtype).contiguous()
    cos, sin = rope_tables(seqlen, head_dim, rope_base, dq.device)
    out = torch.empty((bsz, basis, seqlen, channels), device=dq.device, dtype=dq.dtype)
    with _lib.device_guard(out.device):
        status = _lib.load().lbi_attn_qkv_conv_pullback(
            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), cos.data_ptr(), sin.data_ptr(), weight.data_ptr(),
            out.data_ptr(), bsz, basis, seqlen, heads, n_kv_heads, head_dim, int(bool(rope_interleaved)),
            weight.shape[-1], _lib.dtype_code(out.dtype), _stream(out))
    _lib.check(status, "lbi_attn_qkv_conv_pullback")
    return out


#: widest RMSNorm and longest convolution filter the parameter-gradient kernels take
NORM_GRAD_MAX_WIDTH = 2048
CONV_GRAD_MAX_TAPS = 8


def rmsnorm_weight_grad(g_out: torch.Tensor, x: torch.Tensor, eps: float) -> torch.Tensor:
    """Gradient of an RMSNorm weight, fp32 ``[D]``: ``g_out [..., D]`` (in the weight dtype) summed over all rows
    against the normalised input, with ``x [..., D]`` (weight dtype or fp32) rounded to the weight dtype first and
    the normalised value rounded again, as the forward does (reference backbones/transformer/block.py:18-23)."""
    _require_cuda(g_out, x)
    width = g_out.shape[-1]
    if x.shape[-1] != width or x.numel() != g_out.numel():
        raise ValueError("rmsnorm_weight_grad: g_out and x must hold the same rows of the same width")
    if x.dtype not in (g_out.dtype, torch.float32):
        raise ValueError("rmsnorm_weight_grad: x must be in the dtype of g_out or fp32")
    g_out, x = g_out.contiguous(), x.contiguous()
    rows = g_out.numel() // width
    out = torch.empty(width, device=g_out.device, dtype=torch.float32)
    lib = _lib.load()
    with _lib.device_guard(out.device):
        need = int(lib.lbi_rmsnorm_weight_grad_workspace_bytes(rows, width))
        workspace = torch.empty(max(need, 16), device=out.device, dtype=torch.uint8)
        status = lib.lbi_rmsnorm_weight_grad(g_out.data_ptr(), x.data_ptr(), out.data_ptr(), workspace.data_ptr(),
                                             workspace.numel(), rows, width, float(eps), _lib.dtype_code(g_out.dtype),
                                             _lib.dtype_code(x.dtype), _stream(out))
    _lib.check(status, "lbi_rmsnorm_weight_grad")
    return out


def causal_conv1d_weight_grad(g_out: torch.Tensor, x: torch.Tensor, ksize: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Weight ``[C, 1, k]`` and bias ``[C]`` gradients (fp32) of the depthwise causal convolution for
    ``g_out, x [B, T, C]``: ``g_w[c, 0, j] = sum_{b, t} g_out[b, t, c] x[b, t - (k-1-j), c]``."""
    _require_cuda(g_out, x)
    if g_out.dim() != 3 or x.shape != g_out.shape or x.dtype != g_out.dtype:
        raise ValueError("causal_conv1d_weight_grad: g_out and x must share shape [B, T, C] and dtype")
    bsz, seqlen, channels = g_out.shape
    g_out, x = g_out.contiguous(), x.contiguous()
    out = torch.empty(channels * ksize + channels, device=g_out.device, dtype=torch.float32)
    lib = _lib.load()
    with _lib.device_guard(out.device):
        need = int(lib.lbi_causal_conv1d_weight_grad_workspace_bytes(bsz, seqlen, channels, ksize))
        workspace = torch.empty(max(need, 16), device=out.device, dtype=torch.uint8)
        status = lib.lbi_causal_conv1d_weight_grad(g_out.data_ptr(), x.data_ptr(), out.data_ptr(), workspace.data_ptr(),
                                                   workspace.numel(), bsz, seqlen, channels, ksize,
                                                   _lib.dtype_code(g_out.dtype), _stream(out))
    _lib.check(status, "lbi_causal_conv1d_weight_grad")
    return out[:channels * ksize].view(channels, 1, ksize), out[channels * ksize:]


#: rows below which the transposed copy of the weight costs more than the faster product form gains
_TRANSPOSED_COPY_MIN_ROWS = 65536

#: Multiply-adds and results up to which a product runs on the package's own kernel.  A call of the library takes 18 us of
#: host time, one of this kernel 7; on the GPU (bf16, M x K x N, this kernel and the library): 512 x 256 x 1024 3.8 and 5.2 us,
#: 2048 x 2048 x 256 9.0 and 11.8, 1000 x 1536 x 768 9.7 and 10.8, 3001 x 1000 x 520 14.8 and 15.5, 4096 x 256 x 1024 9.2 and 8.4;
#: past the lines 8192 x 256 x 1024 15.4 and 11.7, 4096 x 512 x 2048 21.5 and 15.5; forward products: 500 x 768 x 2304
#: 8.7 and 8.2, 2000 x 512 x 1024 7.4 and 7.9.
_SMALL_PRODUCT = 3 << 29
_SMALL_PRODUCT_RESULTS = 1 << 22

#: Terms of a sum up to which it does: a tile of results is one workgroup's, which takes 0.2 us per 64 terms (0.25 in a gradient)
#: however few tiles there are, while the library cuts long sums.  Whole calls, us, this kernel and the library: 256 x 4096 x 256 13.6 and
#: 17.7, 512 x 6144 x 768 20.5 and 17.7 (among a parameter VJP's other calls, which wait for the host, still the better: d_model 768, B=1
#: T=205 515 and 556 for all of it), 256 x 8192 x 256 24.1 and 17.7, 128 x 65536 x 128 178 and 104.  Gradients, in a block that is one native call, for which
#: the library is slower still: 64 x 16384 x 64 65 and 86, 128 x 16384 x 128 66 and 120.
_SMALL_PRODUCT_TERMS = 6144
_SMALL_GRADIENT_TERMS = 16384


#: how the operands of ``lbi_small_product`` lie
_ROWS_BY_WEIGHT, _GRADIENT, _FORWARD = 0, 1, 2

#: looked at before anything else: the shapes of a product cost a microsecond to take apart
_SMALL_PRODUCT_TYPES = (torch.float16, torch.bfloat16)


def _small_product_size(height: int, width: int, inner: int, form: int, times: int = 1) -> bool:
    long_sums = form == _GRADIENT and min(height, width) >= 64
    return (0 < height * width * inner <= times * _SMALL_PRODUCT and height * width <= times * _SMALL_PRODUCT_RESULTS
            and inner <= (_SMALL_GRADIENT_TERMS if long_sums else _SMALL_PRODUCT_TERMS)
            and width % 8 == 0 and (height if form == _GRADIENT else inner) % 8 == 0
            # what the kernel's 32-bit offsets span, its tiles and the chunks asked for ahead included
            and (max(height, width) + 64) * (inner + 256) < 1 << 30)


def _is_small_product(a: torch.Tensor, w: torch.Tensor, height: int, width: int, inner: int, form: int) -> bool:
    return (a.dtype in _SMALL_PRODUCT_TYPES and w.dtype == a.dtype and w.device == a.device
            and _small_product_size(height, width, inner, form)
            and a.is_contiguous() and w.is_contiguous() and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def small_product(a: torch.Tensor, w: torch.Tensor, out: torch.Tensor, height: int, width: int, inner: int, form: int,
                  seqlen: int = 1, head_dim: int | None = None) -> torch.Tensor:
    """``out`` filled with ``a w``, ``a^T w`` or ``a w^T`` (``form``), ``[height, width]`` with ``inner`` terms a sum; with
    ``head_dim`` as ``[height / seqlen, width / head_dim, seqlen, head_dim]``."""
    _require_cuda(a, w, out)
    with _lib.device_guard(a.device):
        status = _lib.load().lbi_small_product(a.data_ptr(), w.data_ptr(), out.data_ptr(), height, width, inner, form, seqlen,
                                               head_dim or width, _lib.dtype_code(a.dtype), _stream(a))
    _lib.check(status, "lbi_small_product")
    return out


#: Results and multiply-adds up to which a weight gradient runs on the package's own kernels, the library's product not cutting its long
#: sums (us, 8192 rows, own and library): 768 x 768 22 and 57, 768 x 3072 60 and 96, 6144 x 768 95 and 114; past the lines 2048 x 4096 165 and 132,
#: 1024 x 4096 with 32768 rows 342 and 291.
_WEIGHT_GRADIENT_RESULTS = 5 << 20
_WEIGHT_GRADIENT = 3 << 34


def _is_weight_gradient(g: torch.Tensor, x: torch.Tensor) -> bool:
    """Whether ``lbi_weight_gradient`` takes ``g^T x``."""
    if g.dtype not in _SMALL_PRODUCT_TYPES or x.dtype != g.dtype or x.device != g.device or x.shape[0] != g.shape[0]:
        return False
    (rows, height), width = g.shape, int(x.shape[1])
    return (0 < height * width <= _WEIGHT_GRADIENT_RESULTS and 0 < height * width * rows <= _WEIGHT_GRADIENT and height % 8 == 0 and width % 8 == 0
            # what the kernels' 32-bit offsets span, the steps asked for ahead included
            and (max(height, width) + 128) * (rows + 256) < 1 << 30
            and g.is_contiguous() and x.is_contiguous() and g.data_ptr() % 16 == 0 and x.data_ptr() % 16 == 0)


def weight_gradient(g: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """``g^T x`` for ``g [rows, M]`` and ``x [rows, N]`` of one 16-bit type, sums in fp32."""
    _require_cuda(g, x)
    rows, height, width = int(g.shape[0]), int(g.shape[1]), int(x.shape[1])
    out = g.new_empty(height, width)
    lib = _lib.load()
    with _lib.device_guard(g.device):
        need = int(lib.lbi_weight_gradient_workspace_bytes(height, width, rows))
        workspace = torch.empty(need, device=g.device, dtype=torch.uint8) if need else None
        status = lib.lbi_weight_gradient(g.data_ptr(), x.data_ptr(), out.data_ptr(), None if workspace is None else workspace.data_ptr(), need,
                                         height, width, rows, _lib.dtype_code(g.dtype), _stream(g))
    _lib.check(status, "lbi_weight_gradient")
    return out


def _rows_product(g: torch.Tensor, weight: torch.Tensor, head_dim: int | None = None) -> torch.Tensor | None:
    """``g [B,P,T,K] @ weight [K,N]``, with ``head_dim`` as ``[B,P,N/head_dim,T,head_dim]``; ``None`` where it is not a small
    product."""
    if g.dtype not in _SMALL_PRODUCT_TYPES:
        return None
    bsz, basis, seqlen, inner = g.shape
    rows, width = bsz * basis * seqlen, int(weight.shape[1])
    if weight.shape[0] != inner or not _is_small_product(g, weight, rows, width, inner, _ROWS_BY_WEIGHT):
        return None
    if head_dim is None:
        return small_product(g, weight, g.new_empty(bsz, basis, seqlen, width), rows, width, inner, _ROWS_BY_WEIGHT)
    out = g.new_empty(bsz, basis, width // head_dim, seqlen, head_dim)
    return small_product(g, weight, out, rows, width, inner, _ROWS_BY_WEIGHT, seqlen, head_dim)


def _apply_transposed(g: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``g @ weight`` for ``weight [out, in]``: the pullback of ``y = x weight^T``.  For tall ``g`` it is issued as
    the library's ``A B^T`` form on a transposed copy of the (small) weight, which is its faster path for these
    products; for fewer rows (the single direction of a parameter VJP) the copy is not worth it, and for few ones the
    library's call is what takes longest."""
    if weight.dtype != g.dtype:
        # a forward run under autocast multiplied by the weight cast to the compute dtype; so does its pullback
        weight = weight.to(g.dtype)
    small = _rows_product(g, weight)
    if small is not None:
        return small
    if g.numel() // g.shape[-1] < _TRANSPOSED_COPY_MIN_ROWS:
        return torch.matmul(g, weight)
    return torch.nn.functional.linear(g, weight.t().contiguous())


def _apply_transposed_to_heads(g: torch.Tensor, weight: torch.Tensor, n_heads: int, head_dim: int) -> torch.Tensor:
    """``g @ weight`` as ``[B,P,H,T,Dh]``."""
    if weight.dtype != g.dtype:
        weight = weight.to(g.dtype)
    if head_dim % 4 == 0 and weight.shape[1] == n_heads * head_dim:
        small = _rows_product(g, weight, head_dim)
        if small is not None:
            return small
    return attn_heads_split(_apply_transposed(g, weight), n_heads, head_dim)


def _rows(t: torch.Tensor) -> torch.Tensor:
    return t.reshape(-1, t.shape[-1])


def _linear_grads(sink: dict, linear: Any, g_out: torch.Tensor, x: torch.Tensor) -> None:
    """Weight (and bias) gradient of ``y = x W^T + b`` for the single direction in ``g_out [B,1,T,O]``."""
    g2 = _rows(g_out)
    x2 = _rows(x).to(g2.dtype)
    grad = weight_gradient(g2, x2) if _is_weight_gradient(g2, x2) else torch.matmul(g2.t(), x2)
    sink[id(linear.weight)] = grad.to(linear.weight.dtype)
    bias = getattr(linear, "bias", None)
    if bias is not None:
        sink[id(bias)] = g2.float().sum(dim=0).to(bias.dtype)


def _norm_weight_grad(sink: dict, norm: Any, g_out: torch.Tensor, x: torch.Tensor) -> None:
    """Gradient of the RMSNorm weight: sum over rows of g_out o normalised(x), with x rounded to
    the weight dtype first and the normalised value rounded again, as the forward does
    (reference backbones/transformer/block.py:18-23)."""
    wdtype = norm.weight.dtype
    width = x.shape[-1]
    if g_out.dtype == wdtype and x.dtype in (wdtype, torch.float32) and width % 4 == 0 and width <= NORM_GRAD_MAX_WIDTH:
        sink[id(norm.weight)] = rmsnorm_weight_grad(g_out, x, norm.eps).to(wdtype)
        return
    # widths the kernel does not take: the same sum with torch operations on the device
    xf = x.to(wdtype).float()
    normed = (xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + norm.eps)).to(wdtype).float()
    sink[id(norm.weight)] = (_rows(g_out).float() * _rows(normed)).sum(dim=0).to(wdtype)


def _conv_grads(sink: dict, conv: Any, g_out: torch.Tensor, x_pre: torch.Tensor) -> None:
    """Depthwise causal convolution: g_w[c, j] = sum_{b,t} g_out[b,t,c] x_pre[b, t + j - (k-1), c]."""
    ksize = conv.weight.shape[-1]
    if ksize <= CONV_GRAD_MAX_TAPS and x_pre.dtype == g_out.dtype:
        g_weight, g_bias = causal_conv1d_weight_grad(g_out[:, 0], x_pre, ksize)
        sink[id(conv.weight)] = g_weight.to(conv.weight.dtype)
        if getattr(conv, "bias", None) is not None:
            sink[id(conv.bias)] = g_bias.to(conv.bias.dtype)
        return
    # longer filters: the same sums with torch operations on the device
    g = g_out[:, 0].float()
    x = x_pre.float()
    seqlen = g.shape[1]
    cols = []
    for j in range(ksize):
        shift = ksize - 1 - j
        if shift >= seqlen:
            cols.append(torch.zeros(g.shape[-1], device=g.device))
        else:
            cols.append((g[:, shift:] * x[:, :seqlen - shift]).sum(dim=(0, 1)))
    sink[id(conv.weight)] = torch.stack(cols, dim=-1).unsqueeze(1).to(conv.weight.dtype)
    if getattr(conv, "bias", None) is not None:
        sink[id(conv.bias)] = g.sum(dim=(0, 1)).to(conv.bias.dtype)


#: How many times a small product's multiply-adds and results one of a native layer may have: the library is up to twice as fast on those
#: last ones, and the layer still the faster for the host time that it doesn't wait for.  Whole calls, us, launch by launch / native
#: up to 1, 2, 3, 5 times: parameter VJP d_model 768, 2 layers, B=1 T=258 577 / 619, 355, 356, 354; d_model 512, 1 layer, B=2 T=1024
#: 321 / 325, 325, 289, 289; region pullback d_model 512, 1 layer, B=2 T=65 P=9 129 / 130, 80, 79, 79; d_model 256, 2 layers, B=5 T=128
#: P=24 281 / 292, 292, 281, 329; d_model 256, 2 layers, B=1 T=128 P=16 185 / 115 and the same on.
_NATIVE_TIMES = 3


def _lie_ready(dtype: torch.dtype, device: torch.device, tensors: tuple) -> bool:
    """Whether the native layer can take these tensors as they lie."""
    for t in tensors:
        if t.dtype is not dtype or t.data_ptr() & 15 or not t.is_contiguous() or t.device != device:
            return False
    return True


def _native_layer(block: Any, layer_cache: Any, g_hidden: torch.Tensor | None, g_residual: torch.Tensor, want_branch: bool,
                  param_grads: dict | None) -> tuple[torch.Tensor, torch.Tensor | None] | None:
    """:func:`_layer_input_pullback` as one native call (``lbi_region_layer_pullback``: the same launches without the host time
    between them), for 16-bit blocks whose products are all small ones; ``None`` for others.  Nothing is updated in place."""
    attn, mlp = block.attn, block.mlp
    a_cache, m_cache = layer_cache.attention, layer_cache.mlp
    q = a_cache.q_rope
    dtype, device = q.dtype, q.device
    if dtype not in _SMALL_PRODUCT_TYPES or attn.d_conv <= 0 or q.dim() != 4:
        return None
    bsz, basis, g_len, dim = g_residual.shape
    seqlen = q.shape[2]
    rows, fc1_output = bsz * basis * seqlen, m_cache.fc1_output
    # most calls that are not taken leave here: the largest product is not a small one, or its sums are too long
    if fc1_output.shape[-1] > _SMALL_PRODUCT_TERMS or rows * dim * fc1_output.shape[-1] > _NATIVE_TIMES * _SMALL_PRODUCT:
        return None
    heads, kv_heads, head_dim = attn.n_heads, attn.n_kv_heads, attn.head_dim
    conv = attn.conv1d.weight
    hidden, q_width, packed = fc1_output.shape[-1] // 2, heads * head_dim, (heads + 2 * kv_heads) * head_dim
    # the products, and the attention that runs without copies (the rule of attention_input_pullback_basis)
    g_rows = rows if g_len == seqlen else bsz * basis
    if not (_small_product_size(rows, dim, 2 * hidden, _ROWS_BY_WEIGHT, _NATIVE_TIMES) and _small_product_size(g_rows, hidden, dim, _ROWS_BY_WEIGHT, _NATIVE_TIMES)
            and _small_product_size(rows, q_width, dim, _ROWS_BY_WEIGHT, _NATIVE_TIMES) and _small_product_size(rows, dim, packed, _ROWS_BY_WEIGHT, _NATIVE_TIMES)):
        return None
    wide_dim = next((w for w in _MFMA_HEAD_DIMS if w >= head_dim), 0)
    single_launch = seqlen <= _SINGLE_LAUNCH_MAX_SEQ.get(wide_dim, 0)
    if wide_dim == 0 or head_dim % 8 or heads % kv_heads or not (single_launch or seqlen > _MFMA_SEQ_MULTIPLE // 2):
        return None
    attn_edge = wide_dim != head_dim or not (single_launch or seqlen % _MFMA_SEQ_MULTIPLE == 0)
    fc1, fc2, out_proj, in_proj, norm1, norm2 = (mlp.fc1.weight, mlp.fc2.weight, attn.out_proj.weight, attn.in_proj.weight,
                                                 block.norm.weight, block.norm2.weight)
    x1, x2, q, k, v = (t.contiguous() for t in (a_cache.norm_input, m_cache.norm_input, q, a_cache.k_expanded, a_cache.v_expanded))
    taps = conv.shape[-1]
    positions, matrix = (bsz, seqlen, dim), (bsz, heads, seqlen, head_dim)
    if not (taps <= FUSED_CONV_MAX_TAPS and conv.shape == (packed, 1, taps) and fc1_output.shape == (bsz, seqlen, 2 * hidden)
            and q.shape == matrix and k.shape == matrix and v.shape == matrix
            and x1.shape == positions and x2.shape == positions and norm1.shape == (dim,) and norm2.shape == (dim,)
            and fc1.shape == (2 * hidden, dim) and fc2.shape == (dim, hidden) and out_proj.shape == (dim, q_width)
            and in_proj.shape == (packed, dim) and (g_len == seqlen or g_len == 1)
            and g_residual.device == device
            and _lie_ready(dtype, device, (fc1_output, q, k, v, fc1, fc2, out_proj, in_proj, norm1,
                                           norm2, conv))
            and (g_hidden is None or _lie_ready(dtype, device, (g_hidden,)))
            and x1.dtype in (dtype, torch.float32) and _lie_ready(x1.dtype, device, (x1,))
            and x2.dtype in (dtype, torch.float32) and _lie_ready(x2.dtype, device, (x2,))
            and g_residual.dtype is torch.float32 and g_residual.is_contiguous() and g_residual.data_ptr() & 15 == 0):
        return None
    inputs: tuple = ()
    if param_grads is not None:
        inputs = (m_cache.down_input, m_cache.norm_output, a_cache.out_proj_input, a_cache.norm_output)
        if not (basis == 1 and g_len == seqlen and dim % 4 == 0 and dim <= NORM_GRAD_MAX_WIDTH
                and all(getattr(linear, "bias", None) is None for linear in (mlp.fc1, mlp.fc2, attn.out_proj, attn.in_proj, attn.conv1d))
                and inputs[0].shape == (bsz, seqlen, hidden) and inputs[1].shape == positions
                and inputs[2].shape == (bsz, seqlen, q_width) and inputs[3].shape == positions
                and _lie_ready(dtype, device, inputs)
                and _small_product_size(dim, hidden, rows, _GRADIENT, _NATIVE_TIMES) and _small_product_size(2 * hidden, dim, rows, _GRADIENT, _NATIVE_TIMES)
                and _small_product_size(dim, q_width, rows, _GRADIENT, _NATIVE_TIMES) and _small_product_size(packed, dim, rows, _GRADIENT, _NATIVE_TIMES)
                and _small_product_size(rows, packed, dim, _FORWARD, _NATIVE_TIMES)):
            return None
    scale = attn.softmax_scale if attn.softmax_scale is not None else 1.0 / math.sqrt(head_dim)
    cos, sin = rope_tables(seqlen, head_dim, attn.rope_base, device)
    g_input = torch.empty((bsz, basis, seqlen, dim), device=device, dtype=torch.float32)
    branch = torch.empty((bsz, basis, seqlen, dim), device=device, dtype=dtype) if want_branch else None
    grads = [torch.empty(w.shape, device=device, dtype=dtype) for w in (fc2, fc1, out_proj, in_proj, norm2, norm1, conv)] if inputs else ()
    lib = _lib.load()
    layer = _lib.RegionLayer(
        bsz, basis, seqlen, dim, hidden, heads, kv_heads, head_dim, taps,
        _lib.dtype_code(dtype), _lib.dtype_code(x1.dtype), _lib.dtype_code(x2.dtype),
        int(g_len != seqlen), int(bool(attn.rope_interleaved)), int(attn_edge),
        float(block.norm.eps), float(block.norm2.eps), float(scale),
        None if g_hidden is None else g_hidden.data_ptr(), g_residual.data_ptr(),
        fc2.data_ptr(), fc1.data_ptr(), out_proj.data_ptr(), in_proj.data_ptr(), norm2.data_ptr(), norm1.data_ptr(), conv.data_ptr(),
        fc1_output.data_ptr(), x2.data_ptr(), x1.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        cos.data_ptr(), sin.data_ptr(), g_input.data_ptr(), None if branch is None else branch.data_ptr(),
        *(t.data_ptr() for t in inputs), *(t.data_ptr() for t in grads))
    with _lib.device_guard(device):
        need = int(lib.lbi_region_layer_workspace_bytes(ctypes.byref(layer)))
        workspace = torch.empty(need, device=device, dtype=torch.uint8)
        status = lib.lbi_region_layer_pullback(ctypes.byref(layer), workspace.data_ptr(), need, _stream(q))
    _lib.check(status, "lbi_region_layer_pullback")
    if param_grads is not None:
        for param, grad in zip((fc2, fc1, out_proj, in_proj, norm2, norm1, conv), grads):
            param_grads[id(param)] = grad
    return g_input, branch


def _layer_input_pullback(block: Any, layer_cache: Any, g_hidden: torch.Tensor | None, g_residual: torch.Tensor,
                          kernel_mode: str, want_branch: bool, param_grads: dict | None = None,
                          keep_residual: bool = False) -> tuple[torch.Tensor, torch.Tensor | None]:
    """One block, backwards.  ``g_residual`` (fp32, [B,P,T,D]) is the cotangent of the block's
    residual output and may be updated in place (``[B,P,1,D]``: the same at every position, read only; with
    ``keep_residual`` a full-size one is left untouched too);
    ``g_hidden`` is the cotangent of its hidden output
    in the weight dtype (``None``: equal to ``g_residual``).  Returns the cotangent of
    ``hidden (+ residual)`` at the block input in fp32 and, if ``want_branch``, also rounded to
    the weight dtype (the ``g_hidden`` of the block before).

    With ``param_grads`` (a dict filled as ``id(parameter) -> gradient``; P must be 1) the
    parameter gradients of the block are formed on the way, each from the cotangent at the
    output of its module and the cached input of that module."""
    if kernel_mode == "hip":
        done = _native_layer(block, layer_cache, g_hidden, g_residual, want_branch, param_grads)
        if done is not None:
            return done
    attn, mlp = block.attn, block.mlp
    a_cache, m_cache = layer_cache.attention, layer_cache.mlp
    # Branch cotangents live in the dtype the forward's matrix products ran in, which is what the cached
    # attention operands have: the weights' own dtype, or the autocast dtype of a mixed-precision forward
    # (fp32 master weights, 16-bit products; reference train/runners.py:361), whose weights are cast per use.
    wdtype = a_cache.q_rope.dtype
    if g_hidden is None:
        g_hidden = g_residual.to(wdtype)

    # gated MLP: hidden_out = fc2(up * silu(gate)), [up | gate] = fc1(norm2(res2))
    if param_grads is not None:
        _linear_grads(param_grads, mlp.fc2, g_hidden, m_cache.down_input)
    g_down_input = _apply_transposed(g_hidden, mlp.fc2.weight)
    g_fc1 = gated_mlp_pullback(g_down_input, m_cache.fc1_output)
    del g_down_input
    if param_grads is not None:
        _linear_grads(param_grads, mlp.fc1, g_fc1, m_cache.norm_output)
    g_norm2 = _apply_transposed(g_fc1, mlp.fc1.weight)
    del g_fc1
    if param_grads is not None:
        _norm_weight_grad(param_grads, block.norm2, g_norm2, m_cache.norm_input)
    # res2 feeds norm2 and the residual output
    g_res2, g_attn_out = rmsnorm_pullback(g_norm2, m_cache.norm_input, block.norm2.weight, block.norm2.eps,
                                          g_residual, want_branch=True, keep_residual=keep_residual)
    del g_norm2

    # attention: res2 = out_proj(heads) + res1
    if param_grads is not None:
        _linear_grads(param_grads, attn.out_proj, g_attn_out, a_cache.out_proj_input)
    g_heads = _apply_transposed_to_heads(g_attn_out, attn.out_proj.weight, attn.n_heads, attn.head_dim)
    del g_attn_out
    scale = attn.softmax_scale if attn.softmax_scale is not None else 1.0 / math.sqrt(attn.head_dim)
    dq, dk, dv = attention_input_pullback_basis(a_cache.q_rope, a_cache.k_expanded, a_cache.v_expanded, g_heads,
                                                softmax_scale=float(scale), causal=True, kernel_mode=kernel_mode)
    del g_heads
    if attn.d_conv > 0 and param_grads is None and attn.conv1d.weight.shape[-1] <= FUSED_CONV_MAX_TAPS:
        # nothing needs the cotangent of the convolved projection itself: one pass
        g_qkv = attn_qkv_conv_pullback(dq, dk, dv, attn.conv1d.weight, n_kv_heads=attn.n_kv_heads,
                                       rope_base=attn.rope_base, rope_interleaved=attn.rope_interleaved)
        del dq, dk, dv
    else:
        g_qkv = attn_qkv_pullback(dq, dk, dv, n_kv_heads=attn.n_kv_heads, rope_base=attn.rope_base,
                                  rope_interleaved=attn.rope_interleaved)
        del dq, dk, dv
        if attn.d_conv > 0:
            if param_grads is not None:
                # the cache keeps the projection after the convolution only: redo the projection
                bias = getattr(attn.in_proj, "bias", None)
                x_in, weight = a_cache.norm_output.to(wdtype), attn.in_proj.weight.to(wdtype)
                (bsz, seqlen, inner), width = x_in.shape, int(weight.shape[0])
                if bias is None and weight.shape[1] == inner and \
                        _is_small_product(x_in, weight, bsz * seqlen, width, inner, _FORWARD):
                    x_pre = small_product(x_in, weight, x_in.new_empty(bsz, seqlen, width), bsz * seqlen, width, inner, _FORWARD)
                else:
                    x_pre = torch.nn.functional.linear(x_in, weight, None if bias is None else bias.to(wdtype))
                _conv_grads(param_grads, attn.conv1d, g_qkv, x_pre)
                del x_pre
            g_qkv = causal_conv1d_pullback(g_qkv, attn.conv1d.weight)
    if param_grads is not None:
        _linear_grads(param_grads, attn.in_proj, g_qkv, a_cache.norm_output)
    g_norm1 = _apply_transposed(g_qkv, attn.in_proj.weight)
    del g_qkv
    if param_grads is not None:
        _norm_weight_grad(param_grads, block.norm, g_norm1, a_cache.norm_input)
    return rmsnorm_pullback(g_norm1, a_cache.norm_input, block.norm.weight, block.norm.eps, g_res2,
                            want_branch=want_branch)


def _pull_back_region(backend: Any, cache: Any, cotangent: torch.Tensor, kernel_mode: str,
                      param_grads: dict | None) -> torch.Tensor:
    start, end = cache.layer_range
    device = cache.region_input.device
    # region_output = hidden + residual of the last block: both receive the cotangent
    if param_grads is None and cotangent.shape[2] > 1 and cotangent.stride(2) == 0:
        # an expanded view: the same cotangent at every position (what mean pooling sends back).  The last
        # block's down-projection product then runs on one row per (b, p) and the kernels read [B,P,1,*].
        g = cotangent[:, :, :1].to(device=device, dtype=torch.float32, copy=True).contiguous()
    else:
        g = cotangent.to(device=device, dtype=torch.float32).contiguous()
    # the caller's tensor itself when it already is fp32, contiguous and on the device: the last block then
    # writes its residual sum to a new tensor instead of updating in place
    borrowed = g.data_ptr() == cotangent.data_ptr()
    g_branch = None
    for offset in range(end - start - 1, -1, -1):
        layer_cache = cache.layer_caches[offset]
        block = backend.backbone.blocks[layer_cache.layer_index]
        # hidden and residual at a block input enter only through their sum, so one cotangent
        # (fp32, and its rounded copy for the first product of the block before) is carried
        g, g_branch = _layer_input_pullback(block, layer_cache, g_branch, g, kernel_mode, want_branch=offset > 0,
                                            param_grads=param_grads, keep_residual=borrowed)
        borrowed = False
    return g


def region_input_pullback_basis(backend: Any, cache: Any, output_cotangent_basis: torch.Tensor, *,
                                kernel_mode: str = "hip") -> torch.Tensor:
    """``output_cotangent_basis [B, P, T, D]`` -> region-input cotangents ``[B, P, T, D]``.

    ``backend.backbone.blocks`` and ``cache.layer_caches`` use the attribute names of the
    reference's ``TransformerRegionBackend`` / ``TransformerRegionCache``.
    """
    if output_cotangent_basis.dim() != 4:
        raise ValueError("output_cotangent_basis must have shape [B, P, T, D]")
    if not output_cotangent_basis.is_cuda:
        raise RuntimeError("output_cotangent_basis must be a CUDA tensor (this build has no CPU execution path)")
    start, end = cache.layer_range
    if len(cache.layer_caches) != end - start:
        raise ValueError("cache.layer_caches does not match cache.layer_range")
    if end == start:
        return output_cotangent_basis.detach().clone()
    # the result carries no autograd graph (weights and cache are constants here, as in the reference's extension)
    with torch.no_grad():
        g = _pull_back_region(backend, cache, output_cotangent_basis, kernel_mode, None)
        return g.to(device=output_cotangent_basis.device, dtype=output_cotangent_basis.dtype)


def region_parameter_vjp_with_input_cotangent(backend: Any, cache: Any, output_cotangent: torch.Tensor, *,
                                              kernel_mode: str = "hip") -> tuple[dict[str, torch.Tensor], torch.Tensor]:
    """:func:`region_parameter_vjp` together with the cotangent of the region input ``[B, T, D]`` (fp32) that the
    same backward sweep ends with: what a local-VJP provider needs to carry a region's seed on to the decoder of
    the interface and to the canvas, at no extra cost."""
    if output_cotangent.dim() != 3:
        raise ValueError("output_cotangent must have shape [B, T, D]")
    if not output_cotangent.is_cuda:
        raise RuntimeError("output_cotangent must be a CUDA tensor (this build has no CPU execution path)")
    start, end = cache.layer_range
    if len(cache.layer_caches) != end - start:
        raise ValueError("cache.layer_caches does not match cache.layer_range")
    by_id: dict[int, torch.Tensor] = {}
    if end > start:
        with torch.no_grad():
            g_input = _pull_back_region(backend, cache, output_cotangent.unsqueeze(1), kernel_mode, by_id)[:, 0]
    else:
        g_input = output_cotangent.detach().float()
    out: dict[str, torch.Tensor] = {}
    for name, param in backend.named_parameters():
        if param.requires_grad and id(param) in by_id:  # gradients were formed for the region's blocks only
            out[name] = by_id[id(param)].detach()
    return out, g_input


def region_parameter_vjp(backend: Any, cache: Any, output_cotangent: torch.Tensor, *,
                         kernel_mode: str = "hip") -> dict[str, torch.Tensor]:
    """Parameter gradients of one region for ``output_cotangent [B, T, D]``, keyed by the
    parameter names of ``backend.named_parameters()``.

    ``TransformerLowering.parameter_vjp`` of the reference (backends/transformer.py:76-85;
    autograd version :332-355).  One backward sweep over the cached activations with a single
    direction; every weight gradient is a plain GEMM of the cotangent at a module's output
    with the module's cached input.
    """
    return region_parameter_vjp_with_input_cotangent(backend, cache, output_cotangent, kernel_mode=kernel_mode)[0]


__all__ = [
    "attn_heads_split", "attn_qkv_conv_pullback", "attn_qkv_pullback", "causal_conv1d_pullback",
    "causal_conv1d_weight_grad", "gated_mlp_pullback", "rmsnorm_pullback", "rmsnorm_weight_grad", "region_input_pullback_basis", "region_parameter_vjp", "region_parameter_vjp_with_input_cotangent", "rope_tables",
]
