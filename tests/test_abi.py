"""The C ABI: the built library loads without a GPU and exports what include/lbi_hip.h declares."""
from __future__ import annotations

import ctypes
import re
from pathlib import Path

import pytest

from latent_bounded_interfaces_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "lbi_hip.h"


def _declared_symbols() -> list[str]:
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(lbi_[a-z_0-9]+)\s*\(", text)))


def test_header_declares_entry_points():
    names = _declared_symbols()
    assert {"lbi_suffix_scan", "lbi_suffix_cotangents", "lbi_attn_pullback",
            "lbi_attn_pullback_workspace_bytes", "lbi_last_error", "lbi_abi_version"} <= set(names)


def test_binding_table_matches_header():
    assert sorted(_lib.SYMBOLS) == _declared_symbols()


def test_library_exports_every_declared_symbol():
    if not _lib.LIB_PATH.exists():
        pytest.fail(f"{_lib.LIB_PATH} is not built; run python -m latent_bounded_interfaces_amd.build")
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in _declared_symbols():
        assert hasattr(lib, name), f"{name} missing from liblbi_hip.so"
    assert _lib.load().lbi_abi_version() == _lib.ABI_VERSION


def test_argument_validation_needs_no_gpu():
    """Contract violations are rejected on the host before any HIP call."""
    lib = _lib.load()
    assert lib.lbi_suffix_scan(None, None, -1, 2, 4, _lib.LBI_F32, _lib.LBI_F32, None) == -1
    assert b"negative" in lib.lbi_last_error()
    assert lib.lbi_suffix_scan(None, None, 1, 2, 4, 7, _lib.LBI_F32, None) == -1
    assert b"dtype" in lib.lbi_last_error()
    assert lib.lbi_suffix_scan(None, None, 1, 2, 4, _lib.LBI_F32, _lib.LBI_F32, None) == -1
    assert b"null" in lib.lbi_last_error()
    assert lib.lbi_suffix_scan(None, None, 0, 2, 4, _lib.LBI_F32, _lib.LBI_F32, None) == 0
    assert lib.lbi_last_error() == b""
    assert lib.lbi_suffix_cotangents(None, None, None, 1, 2, 4, _lib.LBI_F32, None) == -1
    # the scan entry with flags: unknown bits, g without cot, misaligned operands
    ok = ctypes.c_void_p(256)
    assert lib.lbi_suffix_scan_ex(ok, None, ok, None, 1, 2, 4, _lib.LBI_BF16, _lib.LBI_F32, 6, None) == -1
    assert b"flag" in lib.lbi_last_error()
    assert lib.lbi_suffix_scan_ex(ok, ok, ok, None, 1, 2, 4, _lib.LBI_BF16, _lib.LBI_F32, 0, None) == -1
    assert b"both" in lib.lbi_last_error()
    assert lib.lbi_suffix_scan_ex(ok, None, ctypes.c_void_p(260), None, 1, 2, 4, _lib.LBI_F32, _lib.LBI_F32,
                                  _lib.LBI_SCAN_EXACT_SUFFIX, None) == -1
    assert b"aligned" in lib.lbi_last_error()
    assert lib.lbi_suffix_scan_ex(None, None, None, None, 0, 2, 4, _lib.LBI_F32, _lib.LBI_F32, 1, None) == 0
    assert lib.lbi_suffix_apply(None, None, None, 1, 2, 4, None) == -1
    assert b"null" in lib.lbi_last_error()
    assert lib.lbi_suffix_apply(None, None, None, -1, 2, 4, None) == -1
    assert lib.lbi_suffix_apply(None, None, None, 0, 2, 4, None) == 0
    odd = ctypes.c_void_p(260)  # not 16-byte aligned
    assert lib.lbi_suffix_apply(odd, odd, odd, 1, 2, 4, None) == -1
    assert b"aligned" in lib.lbi_last_error()


def test_region_and_norm_entry_points_validate_on_the_host():
    lib = _lib.load()
    f32 = _lib.LBI_F32
    assert lib.lbi_rmsnorm_pullback(None, None, None, None, None, None, 1, 1, 1, 8, 1e-5, 0, f32, f32, None) == -1
    assert b"null" in lib.lbi_last_error()
    assert lib.lbi_gated_mlp_pullback(None, None, None, 1, 1, 1, 8, 0, 9, None) == -1
    assert lib.lbi_attn_heads_split(None, None, 1, 1, 1, 1, 8, f32, None) == -1
    one = ctypes.c_void_p(256)  # never dereferenced: every call below is rejected before any launch
    assert lib.lbi_attn_qkv_pullback(one, one, one, one, one, one, 1, 1, 4, 3, 2, 8, 0, f32, None) == -1
    assert b"multiple" in lib.lbi_last_error()
    assert lib.lbi_attn_qkv_conv_pullback(one, one, one, one, one, one, one, 1, 1, 4, 2, 2, 7, 0, 4, f32, None) == -1
    assert b"even head dim" in lib.lbi_last_error()
    assert lib.lbi_attn_qkv_conv_pullback(one, one, one, one, one, one, one, 1, 1, 4, 2, 2, 8, 0, 9, f32, None) == -2
    assert b"above 8" in lib.lbi_last_error()
    assert lib.lbi_causal_conv1d_pullback(one, one, one, 1, 4, 8, 4, f32, None) == -1
    assert b"in-place" in lib.lbi_last_error()
    # spectral / Frobenius norms: LDS-resident sizes need no workspace, larger ones two planes per workgroup
    assert lib.lbi_matrix_norms_workspace_bytes(10, 64) == 0
    assert lib.lbi_matrix_norms_workspace_bytes(10, 88) == 0
    assert lib.lbi_matrix_norms_workspace_bytes(10, 90) == 10 * 2 * 96 * 96 * 4
    assert lib.lbi_matrix_norms_workspace_bytes(5000, 256) == 1024 * 2 * 256 * 256 * 4
    assert lib.lbi_matrix_norms(one, one, one, None, 0, 4, 0, f32, None) == -1
    assert lib.lbi_matrix_norms(one, one, one, None, 0, 4, 256, f32, None) == -4
    assert b"workspace" in lib.lbi_last_error()
    assert lib.lbi_matrix_norms(None, None, None, None, 0, 0, 16, f32, None) == 0
    # parameter gradients that are not matrix products
    assert lib.lbi_rmsnorm_weight_grad_workspace_bytes(8192, 768) == 256 * 768 * 4
    assert lib.lbi_rmsnorm_weight_grad_workspace_bytes(10, 768) == 10 * 768 * 4
    assert lib.lbi_rmsnorm_weight_grad(one, one, one, one, 1 << 30, 4, 6, 1e-5, f32, f32, None) == -2
    assert b"multiple of 4" in lib.lbi_last_error()
    assert lib.lbi_rmsnorm_weight_grad(one, one, one, None, 0, 4, 8, 1e-5, f32, f32, None) == -4
    assert lib.lbi_rmsnorm_weight_grad(one, one, one, one, 1 << 30, 4, 8, 1e-5, f32, _lib.LBI_F16, None) == -2
    assert lib.lbi_causal_conv1d_weight_grad_workspace_bytes(8, 1024, 2304, 4) == 8 * 16 * (2304 * 5) * 4
    assert lib.lbi_causal_conv1d_weight_grad(one, one, one, one, 1 << 30, 1, 4, 8, 9, f32, None) == -2
    assert b"above 8" in lib.lbi_last_error()
    assert lib.lbi_causal_conv1d_weight_grad(one, one, one, None, 0, 1, 4, 8, 4, f32, None) == -4
    # attention: short 16-bit sequences at head dim 64 run as one launch and need no workspace
    f16 = _lib.LBI_F16
    assert lib.lbi_attn_pullback_workspace_bytes(8, 8, 128, 64, 4, f16) == 0
    assert lib.lbi_attn_pullback_workspace_bytes(8, 8, 256, 64, 4, f16) == 0
    assert lib.lbi_attn_pullback_workspace_bytes(8, 8, 77, 64, 4, f16) == 0
    assert lib.lbi_attn_pullback_workspace_bytes(8, 8, 128, 128, 4, f16) == 0
    assert lib.lbi_attn_pullback_workspace_bytes(8, 8, 320, 64, 4, f16) == 4 * (64 * 320 + 256 * 320 + 64 * 320 * 64)
    assert lib.lbi_attn_pullback_workspace_bytes(8, 8, 128, 64, 4, f32) > 0
    assert lib.lbi_attn_pullback(one, one, one, one, one, one, one, None, 0, 8, 8, 320, 64, 4, 0.125, 1, f16, None) == -4
    assert b"workspace" in lib.lbi_last_error()
    # the allocation-free entry rejects, on the host, what its static scratch array cannot hold
    assert lib.lbi_attn_pullback_workspace_bytes(4, 16, 4096, 128, 16, _lib.LBI_BF16) > _lib.ATTN_STATIC_SCRATCH_BYTES
    assert lib.lbi_attn_pullback_static(one, one, one, one, one, one, one, 4, 16, 4096, 128, 16, 0.1, 1,
                                        _lib.LBI_BF16, None) == -4
    assert b"static buffer holds" in lib.lbi_last_error()
    assert lib.lbi_attn_pullback_static(None, one, one, one, one, one, one, 1, 1, 320, 64, 1, 0.1, 1, f16, None) == -1
    assert lib.lbi_attn_pullback_static(None, None, None, None, None, None, None, 0, 1, 320, 64, 1, 0.1, 1, f16, None) == 0
    header = HEADER.read_text()
    assert f"#define LBI_ATTN_STATIC_SCRATCH_BYTES ({_lib.ATTN_STATIC_SCRATCH_BYTES >> 20}u << 20)" in header


def test_attention_edge_entry_validates_on_the_host():
    """What lbi_attn_pullback_edge refuses, and with which status, before any launch; a caller falls back on
    lbi_attn_pullback for LBI_ERR_UNSUPPORTED."""
    lib = _lib.load()
    f16, bf16, f32 = _lib.LBI_F16, _lib.LBI_BF16, _lib.LBI_F32
    one, odd = ctypes.c_void_p(256), ctypes.c_void_p(264)  # never dereferenced

    def call(b, h, t, dh, p, *, causal=1, dtype=bf16, tensors=(one,) * 7, workspace=one, size=1 << 40):
        return lib.lbi_attn_pullback_edge(*tensors, workspace, size, b, h, t, dh, p, 0.1, causal, dtype, None)

    need = lib.lbi_attn_pullback_edge_workspace_bytes(2, 3, 1000, 40, 5, bf16)
    assert need == 4 * (6 * 1024 + 30 * 1024 + 6 * 1024 * 64)
    assert lib.lbi_attn_pullback_edge_workspace_bytes(2, 3, 1000, 80, 5, f16) == 4 * (6 * 1024 + 30 * 1024 + 6 * 1024 * 128)
    for shape, dtype in (((2, 3, 200, 40, 5), bf16), ((2, 3, 128, 80, 5), f16),      # single launch: no workspace
                         ((2, 3, 1000, 44, 5), bf16), ((2, 3, 1000, 136, 5), f16),   # not taken
                         ((2, 3, 1000, 40, 5), f32), ((1, 1, 1 << 24, 64, 1), bf16), ((0, 3, 1000, 40, 5), bf16)):
        assert lib.lbi_attn_pullback_edge_workspace_bytes(*shape, dtype) == 0, (shape, dtype)
    assert call(2, 3, 1000, 44, 5) == -2 and call(2, 3, 1000, 136, 5) == -2 and call(2, 3, 1000, 40, 5, dtype=f32) == -2
    assert call(1, 1, 1 << 24, 64, 1) == -2          # a (b, p, h) slice past 2 GiB
    assert call(2, 3, 1000, 40, 5, causal=0) == -2   # long and non-causal
    assert b"causal" in lib.lbi_last_error()
    for i in range(7):
        assert call(2, 3, 1000, 40, 5, tensors=tuple(odd if j == i else one for j in range(7))) == -1
        assert b"aligned" in lib.lbi_last_error()
        assert call(2, 3, 1000, 40, 5, tensors=tuple(None if j == i else one for j in range(7))) == -1
    assert call(2, 3, 1000, 40, 5, size=need - 1) == -4 and call(2, 3, 1000, 40, 5, workspace=None) == -4
    assert call(2, 3, 1000, 40, 5, workspace=odd) == -4
    assert call(2, 3, -1, 40, 5) == -1 and call(2, 3, 1000, 40, 5, dtype=7) == -1
    assert call(2, 3, 1000, 40, 0, tensors=(None,) * 7) == 0
    header = re.sub(r"\s*\n \* ", " ", HEADER.read_text())
    assert "All seven tensors 16-byte aligned (LBI_ERR_INVALID otherwise" in header


def test_small_products_are_those_that_the_entry_takes():
    """The rule that sends a product to lbi_small_product names no size that the entry refuses (the library forms those), and no
    sum so long that one workgroup takes longer over it than the library."""
    import itertools

    from latent_bounded_interfaces_amd.hip.transformer import region

    lib = _lib.load()
    odd = ctypes.c_void_p(264)  # refused after the sizes: nothing is launched
    sizes = (1, 7, 8, 64, 72, 128, 256, 768, 2048, 4096, 6144, 6152, 16384, 16392, 65536, 1 << 19, 1 << 22, 25_000_000)
    taken = 0
    for form, height, width, inner in itertools.product((0, 1, 2), sizes, sizes, sizes):
        if not region._small_product_size(height, width, inner, form):
            continue
        taken += 1
        assert lib.lbi_small_product(odd, odd, odd, height, width, inner, form, 1, width, _lib.LBI_BF16, None) == -1
        assert b"aligned" in lib.lbi_last_error(), (form, height, width, inner)
        assert inner <= (16384 if form == 1 and min(height, width) >= 64 else 6144)
    assert taken > 300
    assert region._small_product_size(128, 128, 16384, 1) and not region._small_product_size(128, 128, 65536, 1)
    assert not region._small_product_size(8, 8, 25_000_000, 1) and not region._small_product_size(1, 1 << 22, 384, 0)


def test_small_product_statuses():
    """What lbi_small_product refuses, each with its status and before anything is launched; empty results are fine."""
    lib = _lib.load()
    ok, odd = ctypes.c_void_p(256), ctypes.c_void_p(264)  # never dereferenced

    def call(a=ok, w=ok, out=ok, m=64, n=64, k=64, form=0, t=1, dh=64, dtype=_lib.LBI_BF16):
        return lib.lbi_small_product(a, w, out, m, n, k, form, t, dh, dtype, None), lib.lbi_last_error()

    for sizes in (dict(m=-1), dict(n=-8), dict(k=-8), dict(t=0), dict(dh=-4)):
        status, text = call(**sizes)
        assert status == -1 and b"bad size" in text, sizes
    assert call(m=0) == (0, b"") and call(n=0) == (0, b"")
    for name in ("a", "w", "out"):
        status, text = call(**{name: None})
        assert status == -1 and b"null" in text
        status, text = call(**{name: odd})
        assert status == -1 and b"aligned" in text
    for form in (-1, 3):
        status, text = call(form=form)
        assert status == -1 and b"form" in text
    for bad in (dict(dtype=_lib.LBI_F32), dict(dtype=7), dict(k=0), dict(n=68, dh=68), dict(k=60), dict(form=1, m=60),
                dict(form=1, m=64, n=64, k=1 << 25), dict(m=1 << 30)):
        status, text = call(**bad)
        assert status == -2 and b"needs half or bfloat16" in text, bad
    assert call(form=1, k=60, a=odd)[0] == -1   # a gradient sums over any number of rows: refused for its alignment only
    for heads in (dict(dh=0), dict(dh=6), dict(dh=48), dict(t=3)):
        status, text = call(**heads)
        assert status == -1 and b"heads of Dh" in text, heads


def test_weight_gradient_statuses():
    """What lbi_weight_gradient refuses before anything is launched, for sums that are cut and for those that lbi_small_product takes."""
    lib = _lib.load()
    ok, odd = ctypes.c_void_p(256), ctypes.c_void_p(264)  # never dereferenced

    def call(a=ok, w=ok, out=ok, ws=ok, need=1 << 40, m=768, n=768, k=8192, dtype=_lib.LBI_BF16):
        return lib.lbi_weight_gradient(a, w, out, ws, need, m, n, k, dtype, None)

    need = lib.lbi_weight_gradient_workspace_bytes(768, 768, 8192)
    assert need > 0 and need % (128 * 128 * 4 * 36) == 0 and lib.lbi_weight_gradient_workspace_bytes(64, 64, 64) == 0
    assert call(need=need - 1) == call(ws=None) == -4 and b"workspace" in lib.lbi_last_error()
    for k in (64, 8192):
        assert call(m=-1, k=k) == -1 and call(m=0, k=k) == 0
        assert all(call(**{name: bad}, k=k) == -1 for name in ("a", "w", "out") for bad in (None, odd))
        assert all(call(**bad, k=k) == -2 for bad in (dict(m=12), dict(n=12), dict(dtype=_lib.LBI_F32)))
    assert call(k=0) == -2 and call(k=1 << 30) == -2 and call(m=1 << 29, n=1 << 29) == -2


def test_fp32_attention_refuses_what_no_grid_holds():
    """More groups than a grid may have threads for: refused on the host, before a kernel has written anything."""
    lib = _lib.load()
    one = ctypes.c_void_p(256)  # never dereferenced
    need = lib.lbi_attn_pullback_workspace_bytes(1024, 1024, 1, 3, 64, _lib.LBI_F32)
    assert need > 0
    assert lib.lbi_attn_pullback(one, one, one, one, one, one, one, one, need, 1024, 1024, 1, 3, 64, 0.1, 1, _lib.LBI_F32,
                                 None) == -2
    assert b"groups" in lib.lbi_last_error()


def test_wrappers_reject_bad_input_before_touching_the_device():
    import torch

    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks

    with pytest.raises(ValueError, match=r"\[B, K, R, R\]"):
        suffix_scan_pullbacks(torch.zeros(2, 3, 4))
    with pytest.raises(ValueError, match="square"):
        suffix_scan_pullbacks(torch.zeros(2, 3, 4, 5))
    with pytest.raises(RuntimeError, match="CUDA tensor"):
        suffix_scan_pullbacks(torch.zeros(2, 3, 4, 4))


def test_region_layer_statuses():
    lib = _lib.load()
    assert lib.lbi_region_layer_workspace_bytes(None) == 0 and b"null" in lib.lbi_last_error()
    sizes = dict(B=1, P=2, T=64, D=64, hidden=128, H=2, Hkv=1, Dh=32, ksize=4, dtype=_lib.LBI_BF16, norm1_dtype=_lib.LBI_BF16,
                 norm2_dtype=_lib.LBI_F32)
    pointers = {name: 256 for name, kind in _lib.RegionLayer._fields_ if kind is ctypes.c_void_p and not name.startswith("grad_")}

    def status(**changes):
        layer = _lib.RegionLayer(**{**sizes, **pointers, **changes})
        return lib.lbi_region_layer_pullback(ctypes.byref(layer), None, 0, None), lib.lbi_region_layer_workspace_bytes(ctypes.byref(layer))

    assert status()[0] == -4 and status()[1] > 0            # LBI_ERR_WORKSPACE: all is well but the workspace
    for changes in (dict(dtype=_lib.LBI_F32), dict(B=0), dict(T=1 << 31), dict(ksize=9), dict(Hkv=3), dict(Dh=30), dict(T=1 << 28),
                    dict(q=None), dict(g_residual=None), dict(grad_fc2=256), dict(grad_fc2=256, P=1),
                    dict(grad_fc2=256, P=1, g_broadcast_t=1)):
        code, need = status(**changes)
        assert code in (-1, -2) and need == 0, changes

