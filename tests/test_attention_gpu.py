"""Parity of the HIP attention input-pullback against the CPU oracle, through the C ABI (needs the GPU)."""
from __future__ import annotations

import json
import math
from pathlib import Path

import pytest
import torch

from oracle import attention as oattn

pytestmark = pytest.mark.gpu

GOLDEN = json.loads((Path(__file__).parent / "golden" / "attention_known_answers.json").read_text())


def _run(q, k, v, g, device, *, scale, causal, mode="hip"):
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    args = [t.to(device) for t in (q, k, v, g)]
    keep = [t.clone() for t in args]
    out = attention_input_pullback_basis(*args, softmax_scale=scale, causal=causal, kernel_mode=mode)
    torch.cuda.synchronize()
    for a, b in zip(args, keep):
        assert torch.equal(a, b), "input was modified"
    return tuple(t.cpu() for t in out)


def _max_rel(actual, truth):
    """max|diff| / max|truth| over a whole tensor."""
    return float((actual.double() - truth.double()).abs().max() / truth.double().abs().max().clamp_min(1e-30))


@pytest.mark.parametrize("case", ["two_keys_equal", "single_token"])
def test_known_answers(case, device):
    c = GOLDEN[case]
    q, k, v, g = (torch.tensor(c[n], dtype=torch.float32) for n in ("q", "k", "v", "d_out"))
    got = _run(q, k, v, g, device, scale=c["softmax_scale"], causal=c["causal"])
    for name, t in zip(("dq", "dk", "dv"), got):
        assert torch.allclose(t, torch.tensor(c[name]), atol=2e-5), name  # the fp32 bar of the reference tests


# fp32 cases of the reference's tests (tests/test_cuda_attention_pullback.py:62-66, 86-90, 115-119)
# plus ragged ones (T not a multiple of the 16-wide tile, odd head dims, T=1).
FP32_CASES = [
    (101, (2, 3, 5, 4), 2), (103, (1, 2, 4, 3), 3), (117, (1, 2, 4, 16), 3),
    (5, (1, 1, 1, 8), 2), (6, (2, 2, 17, 5), 1), (7, (1, 3, 33, 24), 2), (8, (1, 2, 40, 72), 3),
    (9, (1, 1, 64, 64), 2), (10, (1, 2, 19, 130), 1),
]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("seed,shape,basis", FP32_CASES)
def test_fp32_matches_oracle(seed, shape, basis, causal, device):
    torch.manual_seed(seed)
    q = torch.randn(*shape)
    k = torch.randn_like(q)
    v = torch.randn_like(q)
    g = torch.randn(shape[0], basis, *shape[1:])
    scale = 1.0 / math.sqrt(shape[-1])
    got = _run(q, k, v, g, device, scale=scale, causal=causal)
    want = oattn.attention_pullback_sdpa_loop(q, k, v, g, softmax_scale=scale, causal=causal)
    truth = oattn.attention_pullback_dense(q, k, v, g, softmax_scale=scale, causal=causal, dtype=torch.float64)
    for a, b, c in zip(got, want, truth):
        assert a.shape == g.shape and a.dtype == torch.float32
        assert torch.allclose(a, b, atol=2e-5, rtol=2e-5)  # the reference's fp32 bar
        assert torch.allclose(a.double(), c, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape,basis", [((4, 8, 16, 64), 1), ((4, 8, 17, 64), 1), ((16, 8, 16, 64), 8), ((16, 8, 16, 64), 7),
                                         ((16, 8, 16, 96), 8), ((16, 8, 16, 100), 8), ((16, 32, 16, 32), 1),
                                         ((15, 32, 16, 32), 1), ((1, 2, 48, 33), 2), ((1, 2, 49, 33), 2), ((2, 4, 48, 16), 31),
                                         ((2, 4, 48, 16), 32), ((1, 2, 32, 8), 2), ((16, 16, 40, 33), 5), ((1, 2, 1030, 16), 2),
                                         ((4, 8, 260, 32), 8), ((4, 8, 250, 32), 8)])
def test_fp32_either_side_of_the_scalar_kernels(shape, basis, causal, device):
    """Both sides of the lines between the scalar and the matrix-core kernels and between one and two directions per wave;
    the bound of the test below."""
    q, k, v, g = oattn.make_attention_inputs(*shape, basis, dtype=torch.float32, seed=shape[2])
    scale = 1.0 / math.sqrt(shape[-1])
    got = _run(q, k, v, g, device, scale=scale, causal=causal)
    bound = (shape[2] + 2 * shape[3]) * 2.0 ** -24
    for p in range(basis):   # one direction at a time: the dense formula holds T x T per direction
        truth = oattn.attention_pullback_dense(q, k, v, g[:, p:p + 1], softmax_scale=scale, causal=causal, dtype=torch.float64)
        for name, a, c in zip(("dq", "dk", "dv"), got, truth):
            err = float((a[:, p:p + 1].double() - c).abs().max()) / max(float(c.abs().max()), float(g.abs().max()))
            assert err <= bound, (name, p, err, bound)


# fp32 matrix-core kernels: lengths around the 32-row tiles and the 128-row workgroups, head dims at and between the
# compiled widths (33 and 130: scalar loads / the scalar kernels), direction counts that fill one, two or four waves of a
# workgroup with directions and leave the last group a remainder
FP32_MFMA_CASES = [
    ((1, 2, 31, 32), 1), ((2, 1, 32, 64), 2), ((1, 2, 33, 64), 3), ((1, 1, 128, 64), 4), ((1, 1, 129, 64), 5),
    ((1, 2, 160, 36), 6), ((1, 1, 95, 33), 3), ((1, 1, 64, 96), 1), ((1, 1, 97, 80), 2), ((1, 1, 65, 96), 3),
    ((1, 1, 127, 128), 4), ((1, 1, 225, 128), 1), ((1, 1, 70, 100), 5), ((2, 2, 1, 128), 3), ((1, 2, 258, 64), 9),
    ((1, 3, 200, 32), 8), ((1, 1, 40, 130), 2),
]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape,basis", FP32_MFMA_CASES)
def test_fp32_tile_edges_against_fp64(shape, basis, causal, device):
    q, k, v, g = oattn.make_attention_inputs(*shape, basis, dtype=torch.float32, seed=shape[2] * 131 + basis)
    scale = 1.0 / math.sqrt(shape[-1])
    got = _run(q, k, v, g, device, scale=scale, causal=causal)
    truth = oattn.attention_pullback_dense(q, k, v, g, softmax_scale=scale, causal=causal, dtype=torch.float64)
    bound = (shape[2] + 2 * shape[3]) * 2.0 ** -24  # a rounding per term of the sums over keys and over the head dim
    for name, a, c in zip(("dq", "dk", "dv"), got, truth):
        # against the largest cotangent where a result vanishes (one token: dq = dk = 0)
        err = float((a.double() - c).abs().max()) / max(float(c.abs().max()), float(g.abs().max()))
        assert err <= bound, (name, err, bound)


# more and fewer workgroups than CUs, row tiles and groups either side of one for every CU and of two; the statistics by workgroups of
# 128 queries and of 32
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape,basis", [((16, 17, 40, 32), 1), ((12, 16, 33, 64), 2), ((5, 13, 129, 64), 4), ((3, 11, 250, 64), 8),
                                         ((2, 8, 520, 64), 4), ((1, 1, 1055, 128), 2), ((1, 43, 95, 96), 5)])
def test_fp32_workgroups_and_cus(shape, basis, causal, device):
    q, k, v, g = oattn.make_attention_inputs(*shape, basis, dtype=torch.float32, seed=shape[2] + basis)
    scale = 1.0 / math.sqrt(shape[-1])
    got = _run(q, k, v, g, device, scale=scale, causal=causal)
    truth = oattn.attention_pullback_blocked(q, k, v, g, softmax_scale=scale, causal=causal, dtype=torch.float64)
    bound = (shape[2] + 2 * shape[3]) * 2.0 ** -24  # as above
    for name, a, c in zip(("dq", "dk", "dv"), got, truth):
        err = float((a.double() - c).abs().max()) / max(float(c.abs().max()), float(g.abs().max()))
        assert err <= bound, (name, err, bound)


@pytest.mark.parametrize("offset", [0, 1, 4])   # elements in front of each tensor: whole pieces, single ones, 8-byte pieces
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape,basis", [((1, 2, 31, 32), 1), ((1, 2, 33, 60), 3), ((1, 1, 129, 33), 5), ((1, 1, 161, 96), 3),
                                         ((1, 2, 258, 64), 9), ((2, 1, 95, 100), 2), ((1, 1, 225, 128), 4), ((2, 2, 1, 24), 3),
                                         ((1, 20, 321, 64), 9), ((16, 8, 16, 80), 8)])
def test_half_storage_with_fp32_probabilities(shape, basis, causal, dtype, offset, device):
    """16-bit tensors on the fp32 matrix cores: the bound of the test above and one rounding of the result."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis_static

    inputs = oattn.make_attention_inputs(*shape, basis, dtype=dtype, seed=shape[2] * 131 + basis)
    scale = 1.0 / math.sqrt(shape[-1])

    def placed(t):
        return torch.cat((t.new_zeros(offset), t.reshape(-1))).to(device)[offset:].view(t.shape)

    got = tuple(placed(torch.full_like(inputs[3], float("nan"))) for _ in range(3))
    attention_input_pullback_basis_static(*map(placed, inputs), got, softmax_scale=scale, causal=causal)
    truth = oattn.attention_pullback_dense(*inputs, softmax_scale=scale, causal=causal, dtype=torch.float64)
    eps = (shape[2] + 2 * shape[3]) * 2.0 ** -24
    half_ulp, smallest = (2.0 ** -11, 2.0 ** -25) if dtype == torch.float16 else (2.0 ** -8, 0.0)
    for name, a, c in zip(("dq", "dk", "dv"), got, truth):
        fp32_error = eps * max(float(c.abs().max()), float(inputs[3].double().abs().max()))
        excess = (a.cpu().double() - c).abs() - half_ulp * c.abs()
        assert float(excess.max()) <= fp32_error * (1 + half_ulp) + smallest, (name, float(excess.max()), fp32_error)


@pytest.mark.parametrize("shape,basis", [((1, 2, 1, 32), 1), ((1, 2, 70, 64), 3), ((2, 1, 65, 33), 2), ((1, 1, 130, 128), 2),
                                         ((1, 2, 30, 16), 9)])
def test_fp32_rounding_of_delta_cancels(shape, basis, device):
    """delta is summed from the same P and dP that it is subtracted from.  With one visible key dS is exactly zero; so it is
    with zero keys and one value row repeated over a power of two of positions, where P dP sums without rounding."""
    q, k, v, g = oattn.make_attention_inputs(*shape, basis, dtype=torch.float32, seed=shape[2])
    dq, dk, _ = _run(q, k, v + 10.0, g, device, scale=0.3, causal=True)
    assert torch.equal(dq[:, :, :, 0], torch.zeros_like(dq[:, :, :, 0]))
    if shape[2] == 1:
        assert torch.equal(dk, torch.zeros_like(dk))
    rows = 64
    q, g = (torch.randn(*lead, shape[1], rows, shape[3], generator=torch.Generator().manual_seed(rows))
            for lead in ((shape[0],), (shape[0], basis)))
    v = v[:, :, :1].expand(-1, -1, rows, -1).contiguous()
    _, dk, _ = _run(q, torch.zeros_like(q), v, g, device, scale=0.3, causal=False)
    assert torch.equal(dk, torch.zeros_like(dk))


@pytest.mark.parametrize("where", ["q", "k", "v", "d_out"])
@pytest.mark.parametrize("value", [float("inf"), -float("inf")])
@pytest.mark.parametrize("shape,basis,row", [((1, 2, 70, 64), 3, 37), ((1, 1, 129, 33), 1, 128), ((1, 1, 40, 128), 2, 5),
                                             ((1, 1, 200, 96), 5, 95), ((2, 1, 64, 16), 8, 0)])
def test_fp32_values_out_of_sight_stay_there(shape, basis, row, value, where, device):
    """Under the causal mask a value that is not finite reaches only what may see its row: dQ of the rows behind it,
    dK and dV of the rows before it (and its own); the rest is as with finite values, to rounding."""
    tensors = dict(zip(("q", "k", "v", "d_out"), oattn.make_attention_inputs(*shape, basis, dtype=torch.float32, seed=row)))
    clean = _run(*tensors.values(), device, scale=0.2, causal=True)
    tensors[where][..., row, shape[3] // 2] = value
    got = _run(*tensors.values(), device, scale=0.2, causal=True)
    unseen = {"dq": slice(0, row), "dk": slice(row + 1, None), "dv": slice(row + 1, None)}
    if where in ("k", "v"):   # row `row` spoils every later query, and through them every key up to the last
        unseen["dk"] = unseen["dv"] = slice(0, 0)
    for name, a, b in zip(("dq", "dk", "dv"), got, clean):
        a, b = a[..., unseen[name], :], b[..., unseen[name], :]
        assert torch.allclose(a, b, atol=2e-5, rtol=2e-5), name


def test_fp32_scores_of_minus_infinity(device):
    """Keys whose scores are -inf have P = 0 and get zero gradients, past whole tiles of them and beside rows that only
    fill the last tile."""
    q, k, v, g = (t.abs() for t in oattn.make_attention_inputs(1, 2, 71, 64, 2, dtype=torch.float32, seed=4))
    k[:, :, :40] = float("-inf")
    _, dk, dv = _run(q, k, v, g, device, scale=0.2, causal=False)
    assert torch.isfinite(dk).all() and torch.isfinite(dv).all()
    assert not dk[:, :, :, :40].any() and not dv[:, :, :, :40].any()


# 16-bit storage: the MFMA kernels (T % 64 == 0, Dh in {64, 128}; one fused launch for Dh = 64, T <= 128) and the
# generic ones otherwise.
# (121, (1, 2, 16, 64), P) are the reference's fp16 cases (tests/test_cuda_attention_pullback.py:178-243);
# (8, 8, 128, 64) with P=4 is the reference benchmark shape.
LOWP_CASES = [
    (121, (1, 2, 16, 64), 1), (129, (1, 2, 16, 64), 4), (11, (2, 2, 64, 64), 2), (12, (1, 3, 128, 128), 3),
    (13, (2, 1, 192, 64), 5), (14, (1, 2, 320, 128), 2), (15, (1, 1, 576, 128), 1), (16, (8, 8, 128, 64), 4),
    (17, (1, 2, 96, 64), 2), (18, (1, 1, 64, 32), 2), (19, (1, 2, 256, 64), 9), (20, (1, 1, 448, 64), 16),
    # lengths that are no multiple of 64: causal calls are padded onto the matrix-core kernels
    (21, (2, 2, 100, 64), 3), (22, (1, 1, 1000, 128), 2), (23, (1, 2, 33, 64), 2),
    # head dims below 128 that are not 64: zero-padded onto the matrix-core kernels (with the length, if causal)
    (24, (1, 2, 128, 32), 3), (25, (2, 1, 192, 96), 2), (26, (1, 2, 70, 80), 2), (27, (1, 1, 64, 8), 1),
    (28, (1, 1, 128, 160), 2),  # past 128: generic kernels
    # lengths up to 256 at head dim 64 and up to 128 at head dim 128: the single-launch kernel
    # (so are 11, 12, 13, 16, 17, 19 above and, once padded, the causal runs of 21, 23, 24, 27)
    (29, (1, 2, 32, 64), 3), (30, (3, 1, 128, 64), 1), (31, (2, 3, 96, 64), 5), (32, (1, 2, 160, 64), 2),
    (33, (2, 1, 64, 128), 3), (34, (1, 1, 96, 128), 2), (35, (1, 2, 224, 64), 1), (36, (2, 2, 256, 64), 4),
    # the same kernel at lengths that are no multiple of 32 (zero rows in the last tile, keys past the end masked)
    (37, (1, 2, 1, 64), 2), (38, (2, 1, 255, 64), 3), (39, (1, 2, 127, 128), 2), (40, (1, 1, 31, 64), 1),
    (41, (2, 2, 129, 64), 2), (42, (1, 1, 5, 128), 3),
    # past the single-launch limits with direction counts that leave the kernels a ragged tail: a last dQ group of
    # fewer than 8 (Dh = 64) or 4 (Dh = 128) directions, a last dK/dV group of fewer than 4 (Dh = 64, two directions
    # per wave) or an unpaired last direction (Dh = 128)
    (43, (1, 2, 320, 64), 5), (44, (1, 1, 320, 64), 9), (45, (1, 2, 192, 128), 3), (46, (1, 1, 320, 128), 5),
    (47, (1, 1, 384, 64), 11), (48, (2, 1, 192, 128), 7), (49, (1, 1, 512, 64), 3), (50, (1, 1, 256, 128), 9),
    (51, (1, 2, 320, 64), 6), (52, (2, 1, 384, 64), 7), (53, (1, 3, 576, 64), 4), (54, (1, 1, 320, 64), 2),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("seed,shape,basis", LOWP_CASES)
def test_low_precision_matches_oracle(seed, shape, basis, causal, dtype, device):
    q, k, v, g = oattn.make_attention_inputs(*shape, basis, dtype=dtype, seed=seed)
    scale = 1.0 / math.sqrt(shape[-1])
    got = _run(q, k, v, g, device, scale=scale, causal=causal)
    # fp32 path on the same (already rounded) inputs
    truth = oattn.attention_pullback_blocked(q, k, v, g, softmax_scale=scale, causal=causal, dtype=torch.float32)
    for name, a, c in zip(("dq", "dk", "dv"), got, truth):
        assert a.shape == g.shape and a.dtype == dtype
        assert _max_rel(a, c) <= 2e-2, (name, _max_rel(a, c))  # bar: <= 2e-2 against the fp32 path
        assert torch.allclose(a.float(), c, atol=3e-2 * float(c.abs().max()), rtol=3e-2), name


def test_four_kernel_path_at_short_lengths_in_subprocess(device):
    """LBI_ATTN_SMALL=0 sends short sequences through the four-kernel path; it meets the same bar."""
    import os
    import subprocess
    import sys

    code = (
        "import math, sys, torch; sys.path.insert(0, %r);"
        "from oracle import attention as o;"
        "from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis as f;"
        "worst = 0.0\n"
        "for shape, basis, causal in (((2, 2, 64, 64), 2, True), ((8, 8, 128, 64), 4, True), ((1, 2, 128, 64), 3, False),"
        " ((1, 2, 256, 64), 2, True), ((1, 2, 128, 128), 2, True)):\n"
        "    q, k, v, g = o.make_attention_inputs(*shape, basis, dtype=torch.float16, seed=41)\n"
        "    got = f(q.cuda(), k.cuda(), v.cuda(), g.cuda(), softmax_scale=shape[-1] ** -0.5, causal=causal, kernel_mode='hip')\n"
        "    truth = o.attention_pullback_blocked(q, k, v, g, softmax_scale=shape[-1] ** -0.5, causal=causal, dtype=torch.float32)\n"
        "    for a, c in zip(got, truth):\n"
        "        worst = max(worst, float((a.cpu().double() - c.double()).abs().max() / c.double().abs().max()))\n"
        "print(worst); sys.exit(0 if 0.0 < worst <= 2e-2 else 1)"
    ) % str(Path(__file__).resolve().parents[1])
    env = dict(os.environ, LBI_ATTN_SMALL="0")
    res = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stdout + res.stderr


def test_modes_and_contract(device):
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    q, k, v, g = (t.to(device) for t in oattn.make_attention_inputs(1, 2, 16, 64, 4, dtype=torch.float16, seed=131))
    scale = 0.125
    base = attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode="hip")
    for mode in ("fa2_loop", "simple", "fa2_mma_pblock4"):
        out = attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode=mode)
        assert all(torch.equal(a, b) for a, b in zip(out, base))
    # P limits of the reference's modes (tests/test_cuda_attention_pullback.py:163-173, 281-291)
    for mode in ("fa2_p1", "fa2_mma_p1"):
        with pytest.raises(ValueError, match="== 1"):
            attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode=mode)
        one = attention_input_pullback_basis(q, k, v, g[:, :1], softmax_scale=scale, kernel_mode=mode)
        assert all(torch.equal(a, b[:, :1]) for a, b in zip(one, base))
    g5 = torch.cat([g, g[:, :1]], dim=1)
    with pytest.raises(ValueError, match="<= 4"):
        attention_input_pullback_basis(q, k, v, g5, softmax_scale=scale)
    with pytest.raises(ValueError, match="unknown attention pullback kernel_mode"):
        attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode="nope")
    with pytest.raises(ValueError):
        attention_input_pullback_basis(q, k[:, :1], v, g, softmax_scale=scale)
    with pytest.raises(ValueError):
        attention_input_pullback_basis(q, k, v, g[:, 0], softmax_scale=scale)
    # lowering wrapper (reference tests/test_cuda_attention_pullback.py:294-315)
    low = HipTransformerLowering()
    assert low.name == "hip"
    out = low.attention_input_pullback_basis(q=q, k=k, v=v, output_cotangent_basis=g, softmax_scale=scale)
    assert all(torch.equal(a, b) for a, b in zip(out, base))
    # the default mode is the reference's (backends/transformer_cuda.py:31) with its limit of four directions;
    # "hip" is the mode without one
    with pytest.raises(ValueError, match="<= 4"):
        low.attention_input_pullback_basis(q=q, k=k, v=v, output_cotangent_basis=g5, softmax_scale=scale)
    out = low.attention_input_pullback_basis(q=q, k=k, v=v, output_cotangent_basis=g5, softmax_scale=scale,
                                             kernel_mode="hip")
    assert all(torch.equal(a[:, :4], b) for a, b in zip(out, base))
    with pytest.raises(RuntimeError, match="no CPU execution path"):
        low.input_pullback_basis(backend=None, cache=None, output_cotangent_basis=torch.zeros(1, 1, 2, 3))
    with pytest.raises(ValueError):
        low.input_pullback_basis(backend=None, cache=None, output_cotangent_basis=torch.zeros(1, 2, 3))
    with pytest.raises(RuntimeError, match="no CPU execution path"):
        low.parameter_vjp(backend=None, cache=None, output_cotangent=torch.zeros(1, 2, 3))
    with pytest.raises(ValueError):
        low.parameter_vjp(backend=None, cache=None, output_cotangent=torch.zeros(1, 2, 3, 4))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,basis", [((2, 3, 384, 64), 11), ((1, 2, 320, 128), 7), ((1, 2, 1024, 64), 16)])
def test_results_do_not_depend_on_how_directions_are_grouped(shape, basis, dtype, device):
    """A direction's dQ, dK, dV are the same bits whether it is computed alone, in a pair, or among all directions:
    the kernels group directions (eight or four per dQ workgroup, two per dK/dV workgroup, four at head dim 64 with
    a second direction per wave) only to share the S / P tiles; every direction keeps its own products and sums."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    q, k, v, g = (t.to(device) for t in oattn.make_attention_inputs(*shape, basis, dtype=dtype, seed=77))
    scale = 1.0 / math.sqrt(shape[-1])
    whole = attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode="hip")
    for lo, hi in ((0, 2), (2, 3), (3, 6), (basis - 4, basis), (basis - 1, basis)):
        part = attention_input_pullback_basis(q, k, v, g[:, lo:hi].contiguous(), softmax_scale=scale, kernel_mode="hip")
        for name, a, b in zip(("dq", "dk", "dv"), part, whole):
            assert torch.equal(a, b[:, lo:hi]), (name, lo, hi)


# lengths around the tiles of 32, 64 and 128 positions and past the single launch; head dims of one to sixteen pieces
EDGE_CASES = [((1, 2, 257, 64), 1), ((2, 3, 319, 64), 2), ((1, 3, 1000, 64), 5), ((1, 9, 385, 64), 9),
              ((1, 2, 129, 128), 1), ((2, 1, 191, 128), 3), ((1, 2, 545, 128), 2), ((1, 2, 320, 32), 3),
              ((2, 2, 333, 8), 4), ((1, 2, 384, 56), 1), ((1, 3, 450, 80), 11), ((1, 2, 256, 96), 4),
              ((1, 2, 161, 120), 2), ((2, 2, 48, 32), 3), ((1, 2, 250, 40), 2), ((2, 1, 77, 96), 3), ((1, 1, 1, 72), 2)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,basis", EDGE_CASES)
def test_tiles_padded_on_chip_equal_padded_copies(shape, basis, dtype, device):
    """Zero rows and columns appended by hand give the same bits: the sums are the same, in the same order."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    gen = torch.Generator().manual_seed(31)
    bsz, heads, seqlen, dim = shape
    q, k, v = (torch.randn(*shape, generator=gen).to(dtype).to(device) for _ in range(3))
    g = torch.randn(bsz, basis, *shape[1:], generator=gen).to(dtype).to(device)
    wide = 64 if dim <= 64 else 128
    single = seqlen <= {64: 256, 128: 128}[wide]
    pads = (0, wide - dim, 0, 0 if single else -seqlen % 64)
    for causal in (True, False) if single else (True,):
        got = attention_input_pullback_basis(q, k, v, g, softmax_scale=0.2, causal=causal, kernel_mode="hip")
        want = attention_input_pullback_basis(*(torch.nn.functional.pad(t, pads) for t in (q, k, v, g)),
                                              softmax_scale=0.2, causal=causal, kernel_mode="hip")
        for name, a, b in zip(("dq", "dk", "dv"), got, want):
            assert a.shape == g.shape and torch.equal(a, b[..., :seqlen, :dim]), (name, causal)


@pytest.mark.parametrize("where", ["q", "k", "v", "d_out"])
@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan")])
@pytest.mark.parametrize("shape,basis,row", [((1, 2, 321, 64), 1, -1), ((1, 2, 1000, 64), 5, -1), ((1, 1, 300, 80), 2, -1),
                                             ((1, 1, 333, 40), 9, 100), ((1, 2, 161, 96), 1, 0), ((1, 1, 130, 128), 3, 129)])
def test_padding_on_chip_is_zero_beside_infinities(shape, basis, row, value, where, device):
    """What a tile holds past the end is zero, not a copy of the last row or of its last columns: a value there that is
    not finite gives what it gives in copies padded by hand, infinities and NaN included."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    gen = torch.Generator().manual_seed(77)
    bsz, heads, seqlen, dim = shape
    t = {n: torch.randn(*shape, generator=gen).bfloat16() for n in ("q", "k", "v")}
    t["d_out"] = torch.randn(bsz, basis, *shape[1:], generator=gen).bfloat16()
    if where in ("q", "k"):   # one sign, so that an infinite factor gives scores of +inf or -inf and not NaN throughout
        t = {n: x.abs() for n, x in t.items()}
    t[where][..., row, dim - 1] = value
    t = {n: x.to(device) for n, x in t.items()}
    pads = (0, (64 if dim <= 64 else 128) - dim, 0, -seqlen % 64)
    got = attention_input_pullback_basis(*t.values(), softmax_scale=0.2, causal=True, kernel_mode="hip")
    want = attention_input_pullback_basis(*(torch.nn.functional.pad(x, pads) for x in t.values()), softmax_scale=0.2,
                                          causal=True, kernel_mode="hip")
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        b = b[..., :seqlen, :dim]
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num()), name


def test_long_context_properties(device):
    """bf16, T=4096, Dh=128, P=16 on two (b, h) slices: size-independent checks."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    q, k, v, g = (t.to(device) for t in oattn.make_attention_inputs(1, 2, 4096, 128, 16, dtype=torch.bfloat16, seed=0))
    scale = 1.0 / math.sqrt(128)
    dq, dk, dv = attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode="hip")
    again = attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, kernel_mode="hip")
    assert all(torch.equal(a, b) for a, b in zip((dq, dk, dv), again)), "reruns differ"
    # basis independence: direction p alone gives the same slice
    solo = attention_input_pullback_basis(q, k, v, g[:, 5:6].contiguous(), softmax_scale=scale, kernel_mode="hip")
    for a, b in zip(solo, (dq, dk, dv)):
        assert _max_rel(a[:, 0], b[:, 5].float()) <= 2e-2
    # first query row attends one key: dQ there is zero; P=1 slice equals torch's own attention backward
    assert float(dq[:, :, :, 0].abs().max()) <= 1e-5 * float(dq.abs().max())
    qr, kr, vr = (t.float().requires_grad_(True) for t in (q, k, v))
    out = torch.nn.functional.scaled_dot_product_attention(qr, kr, vr, is_causal=True, scale=scale)
    want = torch.autograd.grad(out, (qr, kr, vr), grad_outputs=g[:, 3].float())
    for name, a, b in zip(("dq", "dk", "dv"), (dq, dk, dv), want):
        assert _max_rel(a[:, 3], b) <= 2e-2, (name, _max_rel(a[:, 3], b))


def test_long_context_full_size_slices_match_oracle(device):
    """The whole long-context call (bf16, B=4, H=16, T=4096, Dh=128, P=16: 64 (b, h) pairs, 1 GiB of cotangents,
    3 GiB of results) run once; the first and the last (b, h) pair, two directions each, against per-direction
    SDPA + autograd of that slice in fp32 on the CPU."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    bsz, heads, seq, hd, basis = 4, 16, 4096, 128, 16
    gen = torch.Generator(device=device).manual_seed(0)
    q, k, v = (torch.randn(bsz, heads, seq, hd, device=device, dtype=torch.bfloat16, generator=gen) for _ in range(3))
    g = torch.randn(bsz, basis, heads, seq, hd, device=device, dtype=torch.bfloat16, generator=gen)
    scale = 1.0 / math.sqrt(hd)
    out = attention_input_pullback_basis(q, k, v, g, softmax_scale=scale, causal=True, kernel_mode="hip")
    torch.cuda.synchronize()
    for (b, h), dirs in (((0, 0), (0, 7)), ((bsz - 1, heads - 1), (basis - 1, 6)), ((2, 5), (9, 12))):
        qs, ks, vs = (t[b:b + 1, h:h + 1].float().cpu() for t in (q, k, v))
        gs = g[b:b + 1, list(dirs), h:h + 1].float().cpu()
        want = oattn.attention_pullback_sdpa_loop(qs, ks, vs, gs, softmax_scale=scale, causal=True)
        for name, a, c in zip(("dq", "dk", "dv"), out, want):
            got = a[b:b + 1, list(dirs), h:h + 1].float().cpu()
            assert _max_rel(got, c) <= 2e-2, (name, b, h, _max_rel(got, c))


# Calls that leave CUs without work and calls that don't, either side of the lines between the numbers of directions per workgroup and
# between the two statistics kernels (head dim 128: 3/4 of the CUs), chains of 1 ... 5 key tiles per wave.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,basis", [((1, 2, 320, 64), 3), ((1, 40, 320, 64), 5), ((2, 3, 576, 64), 7), ((1, 3, 192, 128), 2),
                                         ((1, 1, 448, 128), 9), ((1, 70, 320, 128), 3), ((1, 64, 384, 128), 1), ((1, 65, 384, 128), 4)])
def test_directions_and_statistics_by_size(shape, basis, dtype, causal, device):
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    inputs = oattn.make_attention_inputs(*shape, basis, dtype=dtype, seed=basis)
    q, k, v, d_out = (t.to(device) for t in inputs)
    scale = 1.0 / math.sqrt(shape[-1])
    got = attention_input_pullback_basis(q, k, v, d_out, softmax_scale=scale, causal=causal, kernel_mode="hip")
    want = oattn.attention_pullback_dense(*inputs, softmax_scale=scale, causal=causal, dtype=torch.float32)
    # operands of the second products and results are rounded to the storage type: a few of its units against the largest value
    bar = 4e-3 if dtype == torch.float16 else 3e-2
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        diff = a.float().cpu() - b
        assert float(diff.norm() / b.norm()) <= bar / 2, name
        assert float(diff.abs().max() / b.abs().max()) <= bar, name
    one = attention_input_pullback_basis(q, k, v, d_out[:, basis - 1:].contiguous(), softmax_scale=scale, causal=causal, kernel_mode="hip")
    assert all(torch.equal(a[:, basis - 1:], b) for a, b in zip(got, one))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 2, 320, 64), (1, 2, 384, 128), (1, 70, 320, 128)])
@pytest.mark.parametrize("block", [0, 2, 9])
def test_keys_that_are_nan_show(block, shape, dtype, causal, device):
    """A whole tile of 32 keys that are NaN, wherever it lies among the tiles of a wave: every query that sees one of them has no statistics, and
    with it neither its dQ nor a dK or dV that it takes part in is finite."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    inputs = oattn.make_attention_inputs(*shape, 2, dtype=dtype, seed=block)
    q, k, v, d_out = (t.to(device) for t in inputs)
    k[:, 0, 32 * block:32 * block + 32] = float("nan")
    dq, dk, dv = attention_input_pullback_basis(q, k, v, d_out, softmax_scale=shape[-1] ** -0.5, causal=causal, kernel_mode="hip")
    first = 32 * block if causal else 0
    assert bool(dq[:, :, 0, first:].isnan().all())
    assert bool(dk[:, :, 0].isnan().all()) and bool(dv[:, :, 0].isnan().all())
    assert all(bool(t[:, :, 1:].isfinite().all()) for t in (dq, dk, dv))


# Launches of one to sixteen workgroups a CU, whose order is by length over all heads, heads that fill the eight XCDs or not
@pytest.mark.parametrize("shape,basis", [((3, 13, 640, 64), 3), ((2, 20, 1000, 64), 1), ((4, 24, 1024, 64), 1), ((2, 7, 815, 64), 9),
                                         ((1, 56, 700, 128), 2), ((5, 9, 1100, 96), 1)])
def test_order_of_workgroups_changes_nothing(shape, basis, device):
    """The heads of a call, and the same heads in calls of a few workgroups each."""
    from latent_bounded_interfaces_amd.hip.transformer import attention_input_pullback_basis

    b, h, t, dh = shape
    gen = torch.Generator(device=device).manual_seed(t)
    q, k, v = (torch.randn(shape, generator=gen, device=device).bfloat16() for _ in range(3))
    d_out = torch.randn(b, basis, h, t, dh, generator=gen, device=device).bfloat16()

    def run(rows, heads):
        return attention_input_pullback_basis(*(x[rows, heads].contiguous() for x in (q, k, v)), d_out[rows, :, heads].contiguous(),
                                              softmax_scale=dh ** -0.5, causal=True, kernel_mode="hip")

    whole = run(slice(0, b), slice(0, h))
    for row, head in ((0, 0), (b - 1, h - 1), (b // 2, h // 2), (0, h - 1)):
        alone = run(slice(row, row + 1), slice(head, head + 1))
        for a, c in zip(whole, alone):
            a = a[row:row + 1, :, head:head + 1]
            if dh == 64:
                assert torch.equal(a, c)
            else:  # the statistics' order of summation depends on the heads: results differ by a unit of the storage type
                assert bool(((a.float() - c.float()).abs() <= 2.0 ** -7 * c.float().abs() + 2.0 ** -8 * float(c.float().abs().max())).all())
