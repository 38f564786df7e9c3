"""Region-level input pullback on the GPU (through the C ABI) against autograd of the
CPU restatement of the reference's Transformer region."""
import math

import pytest
import torch
import torch.nn.functional as F

from oracle import transformer_region as oreg

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def _tol(dtype):
    return 2e-5 if dtype == torch.float32 else 2e-2


def _max_rel(a, b):
    return float((a.double() - b.double()).abs().max() / b.double().abs().max().clamp_min(1e-30))


def _vjp(fn, inputs, cotangent):
    inputs = [t.detach().double().requires_grad_(True) for t in inputs]
    out = fn(*inputs)
    return torch.autograd.grad(out, inputs, grad_outputs=cotangent.double())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [32, 30, 768])
def test_rmsnorm_pullback(dtype, dim, device):
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(dim)
    b, p, t = 2, 3, 5
    g = torch.randn(b, p, t, dim).to(dtype)
    x = torch.randn(b, t, dim)  # fp32 residual stream
    w = (1 + 0.1 * torch.randn(dim)).to(dtype)
    res = torch.randn(b, p, t, dim)
    total, branch = region.rmsnorm_pullback(g.to(device), x.to(device), w.to(device), 1e-5, res.clone().to(device),
                                            want_branch=True)
    xr = x.to(dtype)  # the norm runs on the input rounded to the weight dtype

    def fwd(xx):
        return xx * torch.rsqrt(xx.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()

    want = torch.stack([_vjp(fwd, [xr], g[:, i])[0] for i in range(p)], dim=1) + res.double()
    assert total.dtype == torch.float32 and branch.dtype == dtype
    assert _max_rel(total.cpu(), want) <= 2e-5  # fp32 arithmetic on the given (rounded) inputs
    assert _max_rel(branch.cpu(), want) <= _tol(dtype)
    # no residual, fp32 output only
    only, none = region.rmsnorm_pullback(g.to(device), x.to(device), w.to(device), 1e-5, None, want_branch=False)
    assert none is None and _max_rel(only.cpu(), want - res.double()) <= 2e-5


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [4, 256, 260, 1020, 1024, 1028])
def test_rmsnorm_pullback_several_directions_per_wave(dtype, dim, device):
    """Enough tokens for four directions per wave, with a last group of one, at the edges of the register-held widths
    and one past them; one direction alone has to give the same bits."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(dim)
    b, p, t = 2, 5, 1025
    g = torch.randn(b, p, t, dim, device=device).to(dtype)
    x = torch.randn(b, t, dim, device=device)
    w = (1 + 0.1 * torch.randn(dim, device=device)).to(dtype)
    res = torch.randn(b, p, t, dim, device=device)
    total, branch = region.rmsnorm_pullback(g, x, w, 1e-5, res.clone(), want_branch=True)
    xr, wg = x.to(dtype).double().unsqueeze(1), w.double() * g.double()
    r = torch.rsqrt(xr.pow(2).mean(-1, keepdim=True) + 1e-5)
    want = r * wg - xr * r.pow(3) * (xr * wg).mean(-1, keepdim=True) + res.double()
    assert _max_rel(total, want) <= 2e-5 and _max_rel(branch, want) <= _tol(dtype)
    for i in (0, p - 1):
        one, one_branch = region.rmsnorm_pullback(g[-1:, i:i + 1].contiguous(), x[-1:], w, 1e-5,
                                                  res[-1:, i:i + 1].contiguous(), want_branch=True)
        assert torch.equal(one[0, 0], total[-1, i]) and torch.equal(one_branch[0, 0], branch[-1, i])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [24, 27, 3072])
def test_gated_mlp_pullback(dtype, hidden, device):
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(hidden)
    b, p, t = 2, 2, 3
    g = torch.randn(b, p, t, hidden).to(dtype)
    fc1 = (2 * torch.randn(b, t, 2 * hidden)).to(dtype)
    got = region.gated_mlp_pullback(g.to(device), fc1.to(device)).cpu()

    def fwd(f):
        return f[..., :hidden] * F.silu(f[..., hidden:])

    want = torch.stack([_vjp(fwd, [fc1], g[:, i])[0] for i in range(p)], dim=1)
    assert got.dtype == dtype and got.shape == (b, p, t, 2 * hidden)
    assert _max_rel(got, want) <= _tol(dtype)
    assert torch.allclose(got.double(), want, atol=_tol(dtype) * 4, rtol=_tol(dtype) * 4)


# directions of a token in one workgroup and in several, the last with fewer; a dense and a broadcast cotangent
@pytest.mark.parametrize("b,p,t,hidden", [(1, 4, 5, 40), (1, 5, 3, 264), (2, 13, 7, 64), (1, 40, 300, 72), (2, 3, 600, 8)])
@pytest.mark.parametrize("broadcast", [False, True])
def test_gated_mlp_pullback_by_direction(b, p, t, hidden, broadcast, device):
    """A direction's result is the one it has alone, bit for bit."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    gen = torch.Generator().manual_seed(p)
    g = torch.randn(b, p, 1 if broadcast else t, hidden, generator=gen).bfloat16().to(device)
    fc1 = torch.randn(b, t, 2 * hidden, generator=gen).bfloat16().to(device)
    got = region.gated_mlp_pullback(g, fc1)
    for i in range(p):
        assert torch.equal(got[:, i:i + 1], region.gated_mlp_pullback(g[:, i:i + 1].contiguous(), fc1)), i


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,head_dim", [(3, 4), (2, 64), (5, 6)])
def test_heads_split(dtype, heads, head_dim, device):
    from latent_bounded_interfaces_amd.hip.transformer import region

    x = torch.randn(2, 3, 7, heads * head_dim).to(dtype)
    got = region.attn_heads_split(x.to(device), heads, head_dim).cpu()
    assert torch.equal(got, x.view(2, 3, 7, heads, head_dim).permute(0, 1, 3, 2, 4).contiguous())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,head_dim,interleaved",
                         [(4, 4, 8, False), (4, 2, 8, True), (6, 2, 6, False), (3, 1, 2, True), (12, 4, 64, False),
                          (2, 1, 64, True)])
def test_qkv_pullback(dtype, heads, kv_heads, head_dim, interleaved, device):
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(heads * 100 + head_dim)
    b, p, t = 2, 3, 9
    dq, dk, dv = (torch.randn(b, p, heads, t, head_dim).to(dtype) for _ in range(3))
    got = region.attn_qkv_pullback(dq.to(device), dk.to(device), dv.to(device), n_kv_heads=kv_heads, rope_base=100.0,
                                   rope_interleaved=interleaved).cpu()
    rep = heads // kv_heads

    def fwd(qkv):  # [b, t, (H + 2 Hkv) Dh] -> concatenated (q_rope, k_expanded, v_expanded)
        q, k, v = qkv.split((heads * head_dim, kv_heads * head_dim, kv_heads * head_dim), dim=-1)
        q = q.view(b, t, heads, head_dim).transpose(1, 2)
        k = k.view(b, t, kv_heads, head_dim).transpose(1, 2)
        v = v.view(b, t, kv_heads, head_dim).transpose(1, 2)
        # float64 rotation from the same fp32 tables as the kernel
        cos, sin = (c.double() for c in oreg.rope_tables(t, head_dim, 100.0))

        def rot(x):
            if interleaved:
                a, c = x[..., 0::2], x[..., 1::2]
                return torch.stack((a * cos - c * sin, a * sin + c * cos), dim=-1).flatten(-2)
            a, c = x[..., : head_dim // 2], x[..., head_dim // 2:]
            return torch.cat((a * cos - c * sin, a * sin + c * cos), dim=-1)

        return torch.cat((rot(q), rot(k).repeat_interleave(rep, dim=1), v.repeat_interleave(rep, dim=1)), dim=1)

    qkv0 = torch.zeros(b, t, (heads + 2 * kv_heads) * head_dim)
    want = torch.stack([_vjp(fwd, [qkv0], torch.cat((dq[:, i], dk[:, i], dv[:, i]), dim=1))[0] for i in range(p)], dim=1)
    assert got.dtype == dtype and got.shape == want.shape
    assert _max_rel(got, want) <= (1e-6 if dtype == torch.float32 else _tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("channels,ksize,seqlen", [(8, 4, 10), (6, 3, 2), (5, 1, 4), (2304, 4, 7)])
def test_causal_conv1d_pullback(dtype, channels, ksize, seqlen, device):
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(channels + ksize)
    b, p = 2, 2
    g = torch.randn(b, p, seqlen, channels).to(dtype)
    w = torch.randn(channels, 1, ksize).to(dtype)
    got = region.causal_conv1d_pullback(g.to(device), w.to(device)).cpu()

    def fwd(x):  # [b, T, C]
        return F.conv1d(x.transpose(1, 2), w.double(), padding=ksize - 1, groups=channels)[..., :seqlen].transpose(1, 2)

    want = torch.stack([_vjp(fwd, [torch.zeros(b, seqlen, channels)], g[:, i])[0] for i in range(p)], dim=1)
    assert _max_rel(got, want) <= (1e-6 if dtype == torch.float32 else _tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows_shape,dim,wide_x", [((2, 5), 32, True), ((3, 1, 7), 36, False), ((1, 300), 768, True),
                                                  ((4, 130), 2048, False), ((1, 1), 4, True)])
def test_rmsnorm_weight_grad(dtype, rows_shape, dim, wide_x, device):
    """Autograd of the norm's forward (input rounded to the weight dtype, normalised value rounded again, reference
    backbones/transformer/block.py:18-23) with respect to the weight, in fp64 on the rounded values."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(dim + len(rows_shape))
    g = torch.randn(*rows_shape, dim).to(dtype)
    x = torch.randn(*rows_shape, dim) * 1.7
    x = x if wide_x else x.to(dtype)
    got = region.rmsnorm_weight_grad(g.to(device), x.to(device), 1e-5)
    assert got.dtype == torch.float32 and got.shape == (dim,)
    xr = x.to(dtype).float()
    normed = (xr * torch.rsqrt(xr.pow(2).mean(-1, keepdim=True) + 1e-5)).to(dtype)
    want = (g.double() * normed.double()).reshape(-1, dim).sum(0)
    # the normalised value is rounded to the storage type before the sum: a last-place difference of the fp32
    # rsqrt can move single elements by one storage ulp
    assert _max_rel(got.cpu(), want) <= (2e-5 if dtype == torch.float32 else 2e-3)
    again = region.rmsnorm_weight_grad(g.to(device), x.to(device), 1e-5)
    assert torch.equal(got, again)


def test_rmsnorm_weight_grad_contract(device):
    from latent_bounded_interfaces_amd.hip.transformer import region

    g = torch.zeros(2, 3, 8, device=device)
    with pytest.raises(ValueError):
        region.rmsnorm_weight_grad(g, torch.zeros(2, 3, 4, device=device), 1e-5)
    with pytest.raises(ValueError):
        region.rmsnorm_weight_grad(g.half(), torch.zeros(2, 3, 8, device=device, dtype=torch.bfloat16), 1e-5)
    with pytest.raises(RuntimeError, match="multiple of 4"):
        region.rmsnorm_weight_grad(torch.zeros(2, 6, device=device), torch.zeros(2, 6, device=device), 1e-5)
    empty = region.rmsnorm_weight_grad(torch.zeros(0, 8, device=device), torch.zeros(0, 8, device=device), 1e-5)
    assert torch.equal(empty.cpu(), torch.zeros(8))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bsz,seqlen,channels,ksize", [(2, 10, 8, 4), (3, 2, 6, 3), (1, 4, 5, 1), (2, 130, 2304, 4),
                                                      (1, 70, 12, 8), (2, 3, 7, 5)])
def test_causal_conv1d_weight_grad(dtype, bsz, seqlen, channels, ksize, device):
    """Autograd of Conv1d(groups=C, padding=k-1) cut to the first T outputs (reference
    backends/transformer.py:121-122) with respect to weight and bias, in fp64 on the stored values."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(channels + ksize + seqlen)
    g = torch.randn(bsz, seqlen, channels).to(dtype)
    x = torch.randn(bsz, seqlen, channels).to(dtype)
    g_w, g_b = region.causal_conv1d_weight_grad(g.to(device), x.to(device), ksize)
    assert g_w.shape == (channels, 1, ksize) and g_b.shape == (channels,) and g_w.dtype == torch.float32
    w = torch.zeros(channels, 1, ksize, dtype=torch.float64, requires_grad=True)
    b = torch.zeros(channels, dtype=torch.float64, requires_grad=True)
    y = F.conv1d(x.double().transpose(1, 2), w, b, padding=ksize - 1, groups=channels)[..., :seqlen].transpose(1, 2)
    want_w, want_b = torch.autograd.grad(y, (w, b), grad_outputs=g.double())
    assert _max_rel(g_w.cpu(), want_w) <= 2e-5 and _max_rel(g_b.cpu(), want_b) <= 2e-5
    again = region.causal_conv1d_weight_grad(g.to(device), x.to(device), ksize)
    assert torch.equal(g_w, again[0]) and torch.equal(g_b, again[1])


@pytest.mark.parametrize("bsz,seqlen,channels,ksize", [(1, 15, 8, 4), (1, 17, 8, 4), (3, 33, 12, 8), (8, 256, 8, 4), (8, 257, 5, 4), (1, 4095, 4, 3),
                                                      (2, 2049, 4, 4)])
def test_causal_conv1d_weight_grad_by_slab_length(bsz, seqlen, channels, ksize, device):
    """Slabs of 16, 32 and 64 positions, whole and cut, at the lines between them."""
    test_causal_conv1d_weight_grad(torch.float32, bsz, seqlen, channels, ksize, device)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,head_dim,interleaved,ksize,seqlen",
                         [(4, 2, 8, False, 4, 19), (4, 4, 8, True, 3, 8), (3, 1, 6, False, 4, 5), (3, 1, 2, True, 1, 9),
                          (12, 4, 64, False, 4, 33), (2, 1, 64, True, 7, 12), (2, 2, 16, False, 8, 3)])
def test_qkv_conv_pullback_equals_the_two_calls(dtype, heads, kv_heads, head_dim, interleaved, ksize, seqlen, device):
    """The one-pass projection + convolution pullback repeats the arithmetic of the two kernels it replaces (each
    of which is checked against autograd above), through run boundaries, sequence ends and grouped heads."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(heads * 1000 + head_dim * 10 + ksize)
    b, p = 2, 3
    channels = (heads + 2 * kv_heads) * head_dim
    dq, dk, dv = (torch.randn(b, p, heads, seqlen, head_dim).to(dtype).to(device) for _ in range(3))
    weight = torch.randn(channels, 1, ksize).to(dtype).to(device)
    kwargs = dict(n_kv_heads=kv_heads, rope_base=100.0, rope_interleaved=interleaved)
    want = region.causal_conv1d_pullback(region.attn_qkv_pullback(dq, dk, dv, **kwargs), weight)
    got = region.attn_qkv_conv_pullback(dq, dk, dv, weight, **kwargs)
    assert got.dtype == dtype and got.shape == want.shape
    differing = int((got != want).sum())
    if dtype == torch.float32:
        assert differing == 0, f"{differing} elements differ"
    else:
        # same arithmetic, but the compiler may fuse a final multiply-add with the narrowing conversion in one
        # kernel and not in the other: a last-place difference on a few elements in 10^5 is allowed, nothing more
        ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
        assert differing <= max(1, got.numel() // 2000), f"{differing} of {got.numel()} elements differ"
        assert float(((got.float() - want.float()).abs() / want.float().abs().clamp_min(1e-3)).max()) <= ulp


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,head_dim,ksize,interleaved,seqlen",
                         [(4, 4, 64, 4, False, 33), (4, 2, 64, 4, True, 16), (6, 2, 64, 4, False, 47),
                          (8, 2, 64, 4, True, 33), (8, 1, 64, 3, False, 17), (4, 2, 64, 2, False, 31), (3, 3, 64, 3, True, 16),
                          (6, 2, 36, 4, False, 33), (4, 1, 64, 6, False, 20)])
def test_qkv_conv_pullback_many_sequences(dtype, heads, kv_heads, head_dim, ksize, interleaved, seqlen, device):
    """Enough sequences for the long runs (16 positions per thread), with sequences that end in a run of 1, 16 and 15;
    the last sequence alone runs in short ones and has to give the same bits."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(seqlen)
    runs, units_per_run = -(-seqlen // 16), (heads + 2 * kv_heads) * (head_dim // (8 if head_dim % 8 == 0 else 2))
    b, p = 2, 262144 // (2 * runs * units_per_run) + 8
    dq, dk, dv = (torch.randn(b, p, heads, seqlen, head_dim, device=device).to(dtype) for _ in range(3))
    weight = torch.randn((heads + 2 * kv_heads) * head_dim, 1, ksize, device=device).to(dtype)
    kwargs = dict(n_kv_heads=kv_heads, rope_base=100.0, rope_interleaved=interleaved)
    want = region.causal_conv1d_pullback(region.attn_qkv_pullback(dq, dk, dv, **kwargs), weight)
    got = region.attn_qkv_conv_pullback(dq, dk, dv, weight, **kwargs)
    last = region.attn_qkv_conv_pullback(*(t[-1:, -1:].contiguous() for t in (dq, dk, dv)), weight, **kwargs)
    assert torch.equal(last[0, 0], got[-1, -1])
    if dtype == torch.float32:
        assert torch.equal(got, want)
    else:  # a final multiply-add fused with the narrowing in one kernel and not in the other: a last place, rarely
        ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
        assert int((got != want).sum()) <= max(1, got.numel() // 2000)
        assert float(((got.float() - want.float()).abs() / want.float().abs().clamp_min(1e-3)).max()) <= ulp


def test_qkv_conv_pullback_contract(device):
    from latent_bounded_interfaces_amd._lib import LbiLibraryError
    from latent_bounded_interfaces_amd.hip.transformer import region

    dq = torch.randn(1, 1, 2, 4, 8, device=device)
    with pytest.raises(ValueError, match="depthwise"):
        region.attn_qkv_conv_pullback(dq, dq, dq, torch.randn(5, 1, 4, device=device), n_kv_heads=2, rope_base=10.0,
                                      rope_interleaved=False)
    with pytest.raises(LbiLibraryError, match="above 8"):
        region.attn_qkv_conv_pullback(dq, dq, dq, torch.randn(48, 1, 9, device=device), n_kv_heads=2, rope_base=10.0,
                                      rope_interleaved=False)
    with pytest.raises(RuntimeError, match="no CPU execution path"):
        region.attn_qkv_conv_pullback(dq.cpu(), dq.cpu(), dq.cpu(), torch.randn(48, 1, 4), n_kv_heads=2,
                                      rope_base=10.0, rope_interleaved=False)


REGION_CASES = [
    # dim, heads, kv, head_dim, hidden, layers, d_conv, interleaved, B, P, T
    (32, 4, 2, 8, 48, 2, 4, False, 2, 3, 12),
    (24, 3, 3, 8, 40, 1, 0, True, 1, 2, 9),
    (16, 2, 1, 6, 20, 3, 2, False, 2, 2, 5),
]


@pytest.mark.parametrize("case", REGION_CASES)
def test_region_pullback_fp32_matches_autograd(case, device):
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    dim, heads, kv, hd, hidden, layers, d_conv, inter, b, p, t = case
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=kv, head_dim=hd, hidden=hidden, layers=layers,
                                d_conv=d_conv, rope_interleaved=inter, rope_base=1000.0, seed=dim)
    torch.manual_seed(t)
    x = torch.randn(b, t, dim)
    basis = torch.randn(b, p, t, dim)
    _, cpu_cache = backend.forward_region(region_input=x, region_index=0)
    want = oreg.input_pullback_basis_autograd(backend, cpu_cache, basis)

    gpu_backend = backend.to(device)
    with torch.no_grad():
        _, cache = gpu_backend.forward_region(region_input=x.to(device), region_index=0)
    basis_d = basis.to(device)
    got = HipTransformerLowering().input_pullback_basis(backend=gpu_backend, cache=cache,
                                                        output_cotangent_basis=basis_d)
    assert got.shape == basis.shape and got.dtype == basis.dtype and got.is_cuda
    assert _max_rel(got.cpu(), want) <= 2e-5, _max_rel(got.cpu(), want)
    assert torch.equal(basis_d.cpu(), basis) and got.data_ptr() != basis_d.data_ptr()  # the caller's tensor is read only
    assert not got.requires_grad and got.grad_fn is None  # no autograd graph although the weights require grad


@pytest.mark.parametrize("dtype", DTYPES)
def test_kernels_take_position_constant_cotangents(dtype, device):
    """[B,P,1,*] inputs (the same cotangent at every position) give exactly what their expanded copies give."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(5)
    b, p, t, dim, hidden = 2, 3, 7, 40, 24
    g = torch.randn(b, p, t, dim).to(dtype).to(device)
    x = torch.randn(b, t, dim, device=device)
    w = (1 + 0.1 * torch.randn(dim)).to(dtype).to(device)
    res1 = torch.randn(b, p, 1, dim, device=device)
    total, branch = region.rmsnorm_pullback(g, x, w, 1e-5, res1, want_branch=True)
    want_total, want_branch = region.rmsnorm_pullback(g, x, w, 1e-5, res1.expand(b, p, t, dim).contiguous(),
                                                      want_branch=True)
    assert torch.equal(total, want_total) and torch.equal(branch, want_branch)
    assert total.data_ptr() != res1.data_ptr()
    gd1 = torch.randn(b, p, 1, hidden).to(dtype).to(device)
    fc1 = (2 * torch.randn(b, t, 2 * hidden)).to(dtype).to(device)
    got = region.gated_mlp_pullback(gd1, fc1)
    assert torch.equal(got, region.gated_mlp_pullback(gd1.expand(b, p, t, hidden).contiguous(), fc1))
    with pytest.raises(ValueError, match=r"\[B, P, 1, hidden\]"):
        region.gated_mlp_pullback(gd1.expand(b, p, 2, hidden), fc1)
    with pytest.raises(ValueError, match=r"\[B, P, 1, D\]"):
        region.rmsnorm_pullback(g, x, w, 1e-5, torch.zeros(b, p, 2, dim, device=device), want_branch=False)


@pytest.mark.parametrize("case", REGION_CASES)
@pytest.mark.parametrize("dtype", DTYPES)
def test_region_pullback_of_an_expanded_view(case, dtype, device):
    """A stride-0 basis over positions takes the shortened path through the last block; the result is that of
    the dense copy of the same basis (up to the rounding of a product run on fewer rows)."""
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    dim, heads, kv, hd, hidden, layers, d_conv, inter, b, p, t = case
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=kv, head_dim=hd, hidden=hidden, layers=layers,
                                d_conv=d_conv, rope_interleaved=inter, rope_base=1000.0, seed=dim, dtype=dtype).to(device)
    torch.manual_seed(t)
    x = torch.randn(b, t, dim, device=device)
    pooled = torch.randn(b, p, 1, dim, device=device)
    with torch.no_grad():
        _, cache = backend.forward_region(region_input=x, region_index=0)
    lowering = HipTransformerLowering()
    view = pooled.expand(b, p, t, dim)
    assert view.stride(2) == 0
    got = lowering.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=view)
    want = lowering.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=view.contiguous())
    assert got.shape == want.shape == (b, p, t, dim)
    assert _max_rel(got.cpu(), want.cpu()) <= (1e-6 if dtype == torch.float32 else _tol(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("residual_in_fp32", [True, False])
def test_region_pullback_16bit_matches_fp32_path(dtype, residual_in_fp32, device):
    """16-bit weights and activations (MFMA attention path: Dh=64, T=128) against fp32 autograd
    of the same (rounded) weights."""
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    dim, heads, kv, hd, hidden, layers, b, p, t = 128, 2, 1, 64, 256, 2, 2, 5, 128
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=kv, head_dim=hd, hidden=hidden, layers=layers,
                                d_conv=4, residual_in_fp32=residual_in_fp32, dtype=dtype, seed=11)
    torch.manual_seed(12)
    x = torch.randn(b, t, dim).to(dtype)
    basis = torch.randn(b, p, t, dim)
    import copy

    ref_backend = copy.deepcopy(backend).float()  # same rounded weights, fp32 arithmetic
    _, ref_cache = ref_backend.forward_region(region_input=x.float(), region_index=0)
    want = oreg.input_pullback_basis_autograd(ref_backend, ref_cache, basis)

    gpu_backend = backend.to(device)
    with torch.no_grad():
        _, cache = gpu_backend.forward_region(region_input=x.to(device), region_index=0)
    got = HipTransformerLowering().input_pullback_basis(backend=gpu_backend, cache=cache,
                                                        output_cotangent_basis=basis.to(device))
    assert got.dtype == basis.dtype
    assert _max_rel(got.cpu(), want) <= 2e-2, _max_rel(got.cpu(), want)


def test_region_pullback_contract(device):
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    backend = oreg.make_backend(dim=16, n_heads=2, head_dim=8, hidden=16, layers=1, seed=1).to(device)
    x = torch.randn(1, 4, 16, device=device)
    with torch.no_grad():
        _, cache = backend.forward_region(region_input=x, region_index=0)
    low = HipTransformerLowering()
    with pytest.raises(ValueError, match=r"\[B, P, T, D\]"):
        low.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=torch.zeros(1, 4, 16, device=device))
    # linear in the cotangent, and direction p depends on basis[:, p] only
    basis = torch.randn(1, 3, 4, 16, device=device)
    out = low.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=basis)
    one = low.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=basis[:, 1:2])
    assert torch.allclose(out[:, 1:2], one, atol=1e-6)
    twice = low.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=2 * basis)
    assert torch.allclose(twice, 2 * out, atol=1e-5)
    # a zero-layer range is the identity
    cache.layer_range, cache.layer_caches = (0, 0), []
    assert torch.equal(low.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=basis), basis)


@pytest.mark.parametrize("case", REGION_CASES)
@pytest.mark.parametrize("bias", [False, True])
def test_parameter_vjp_fp32_matches_autograd(case, bias, device):
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    dim, heads, kv, hd, hidden, layers, d_conv, inter, b, p, t = case
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=kv, head_dim=hd, hidden=hidden, layers=layers + 1,
                                region_ranges=[(0, 1), (1, layers + 1)], d_conv=d_conv, rope_interleaved=inter,
                                rope_base=1000.0, bias=bias, seed=dim + 1)
    torch.manual_seed(t)
    x = torch.randn(b, t, dim)
    cot = torch.randn(b, t, dim)
    _, cpu_cache = backend.forward_region(region_input=x, region_index=1)
    want = oreg.parameter_vjp_autograd(backend, cpu_cache, cot)

    gpu_backend = backend.to(device)
    with torch.no_grad():
        _, cache = gpu_backend.forward_region(region_input=x.to(device), region_index=1)
    got = HipTransformerLowering().parameter_vjp(backend=gpu_backend, cache=cache, output_cotangent=cot.to(device))
    assert set(got) == set(want) and all(n.startswith("backbone.blocks.") for n in got)
    assert not any(n.startswith("backbone.blocks.0.") for n in got)  # region 1 owns layers 1..
    for name, w in want.items():
        g = got[name].cpu()
        assert g.shape == w.shape and g.dtype == w.dtype
        assert _max_rel(g, w) <= 2e-5, (name, _max_rel(g, w))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_parameter_vjp_16bit_matches_fp32_path(dtype, device):
    import copy

    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    dim, heads, kv, hd, hidden, layers, b, t = 128, 2, 1, 64, 256, 2, 2, 128
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=kv, head_dim=hd, hidden=hidden, layers=layers,
                                d_conv=4, dtype=dtype, seed=13)
    torch.manual_seed(14)
    x = torch.randn(b, t, dim).to(dtype)
    cot = torch.randn(b, t, dim)
    ref_backend = copy.deepcopy(backend).float()
    _, ref_cache = ref_backend.forward_region(region_input=x.float(), region_index=0)
    want = oreg.parameter_vjp_autograd(ref_backend, ref_cache, cot)
    gpu_backend = backend.to(device)
    with torch.no_grad():
        _, cache = gpu_backend.forward_region(region_input=x.to(device), region_index=0)
    got = HipTransformerLowering().parameter_vjp(backend=gpu_backend, cache=cache, output_cotangent=cot.to(device))
    assert set(got) == set(want)
    for name, w in want.items():
        assert got[name].dtype == dtype
        assert _max_rel(got[name].cpu(), w) <= 3e-2, (name, _max_rel(got[name].cpu(), w))


def test_kernels_at_the_end_to_end_scale(device):
    """B=8, P=64, T=1024, d_model 768 / hidden 3072 (up to 3.2e9 elements per tensor, past 2^31): the last batch
    element and direction of every kernel's output equal the same kernel run on that slice alone."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    torch.manual_seed(0)
    b, p, t, heads, hd, dim, hidden = 8, 64, 1024, 12, 64, 768, 3072
    dt = torch.bfloat16
    gd = torch.randn(b, p, t, hidden, device=device, dtype=dt)
    fc1 = torch.randn(b, t, 2 * hidden, device=device, dtype=dt)
    full = region.gated_mlp_pullback(gd, fc1)
    assert torch.equal(full[-1, -1], region.gated_mlp_pullback(gd[-1:, -1:].contiguous(), fc1[-1:])[0, 0])
    del gd, fc1, full
    x = torch.randn(b, t, dim, device=device)
    wn = (1 + 0.1 * torch.randn(dim, device=device)).to(dt)
    gy = torch.randn(b, p, t, dim, device=device, dtype=dt)
    res = torch.randn(b, p, t, dim, device=device)
    tot, br = region.rmsnorm_pullback(gy, x, wn, 1e-5, res.clone(), want_branch=True)
    tot1, br1 = region.rmsnorm_pullback(gy[-1:, -1:].contiguous(), x[-1:], wn, 1e-5, res[-1:, -1:].contiguous(),
                                        want_branch=True)
    assert torch.equal(tot[-1, -1], tot1[0, 0]) and torch.equal(br[-1, -1], br1[0, 0])
    hs = region.attn_heads_split(gy, heads, hd)
    assert torch.equal(hs[-1, -1], gy[-1, -1].view(t, heads, hd).transpose(0, 1))
    del tot, br, res, hs, gy
    dq, dk, dv = (torch.randn(b, p, heads, t, hd, device=device, dtype=dt) for _ in range(3))
    w = torch.randn(3 * heads * hd, 1, 4, device=device, dtype=dt)
    kw = dict(n_kv_heads=heads, rope_base=10000.0, rope_interleaved=False)
    full = region.attn_qkv_conv_pullback(dq, dk, dv, w, **kw)
    part = region.attn_qkv_conv_pullback(*(z[-1:, -1:].contiguous() for z in (dq, dk, dv)), w, **kw)
    assert torch.equal(full[-1, -1], part[0, 0])
    two = region.causal_conv1d_pullback(region.attn_qkv_pullback(dq, dk, dv, **kw), w)
    assert int((two != full).sum()) <= full.numel() // 2000


def test_region_pullback_at_the_end_to_end_layer_shape_matches_oracle(device):
    """Two layers of the end-to-end configuration (d_model 768, 12 heads x 64, hidden 3072, conv 4, T=1024, bf16
    weights and activations, fp32 residual stream) with B=1 and P=4 against fp32 autograd of the CPU restatement
    on the same rounded weights: the values behind the full-size timings, not only their indexing."""
    import copy

    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    dim, heads, hd, hidden, layers, b, p, t = 768, 12, 64, 3072, 2, 1, 4, 1024
    dtype = torch.bfloat16
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=heads, head_dim=hd, hidden=hidden, layers=layers,
                                d_conv=4, residual_in_fp32=True, dtype=dtype, seed=21)
    torch.manual_seed(22)
    x = torch.randn(b, t, dim).to(dtype)
    basis = torch.randn(b, p, t, dim)
    ref_backend = copy.deepcopy(backend).float()
    _, ref_cache = ref_backend.forward_region(region_input=x.float(), region_index=0)
    want = oreg.input_pullback_basis_autograd(ref_backend, ref_cache, basis)
    gpu_backend = backend.to(device)
    with torch.no_grad():
        _, cache = gpu_backend.forward_region(region_input=x.to(device), region_index=0)
    low = HipTransformerLowering()
    got = low.input_pullback_basis(backend=gpu_backend, cache=cache, output_cotangent_basis=basis.to(device))
    assert _max_rel(got.cpu(), want) <= 2e-2, _max_rel(got.cpu(), want)
    # the position-constant form a mean-pooling interface produces (stride-0 view over positions)
    const = torch.randn(b, p, 1, dim)
    want_c = oreg.input_pullback_basis_autograd(ref_backend, ref_cache, const.expand(b, p, t, dim).contiguous())
    got_c = low.input_pullback_basis(backend=gpu_backend, cache=cache,
                                     output_cotangent_basis=const.to(device).expand(b, p, t, dim))
    assert _max_rel(got_c.cpu(), want_c) <= 2e-2, _max_rel(got_c.cpu(), want_c)
    # parameter gradients of the same two layers
    cot = torch.randn(b, t, dim)
    want_p = oreg.parameter_vjp_autograd(ref_backend, ref_cache, cot)
    got_p = low.parameter_vjp(backend=gpu_backend, cache=cache, output_cotangent=cot.to(device))
    assert set(got_p) == set(want_p)
    for name, w in want_p.items():
        assert _max_rel(got_p[name].cpu(), w) <= 3e-2, (name, _max_rel(got_p[name].cpu(), w))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lead,inner,width,head_dim", [
    ((1, 1, 1), 8, 8, 4), ((1, 2, 17), 72, 104, 52), ((2, 3, 11), 256, 64, 32), ((1, 1, 129), 64, 1024, 64),
    ((2, 1, 333), 320, 136, 8), ((1, 5, 64), 448, 256, 128), ((1, 16, 128), 2048, 256, 64), ((1, 1, 3001), 200, 520, 40),
    ((3, 1, 1), 136, 72, 72), ((2, 4, 250), 392, 1032, 24),
])
def test_small_product(lead, inner, width, head_dim, dtype, device):
    """Rows, columns and chunks of the reduction that end inside a tile, both tile heights, one chunk to more than a turn of the
    ring; infinities stay in their row and column."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    gen = torch.Generator().manual_seed(inner + width)
    g = torch.randn(*lead, inner, generator=gen).to(dtype)
    weight = torch.randn(inner, width, generator=gen).to(dtype)
    rows = math.prod(lead)
    truth = g.double() @ weight.double()
    # a rounding per term of the sum, then one of the result
    sums = g.double().abs() @ weight.double().abs()
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = (inner + 1) * 2.0 ** -24 * sums * (1 + half_ulp) + half_ulp * truth.abs() + 2.0 ** -25

    def product(a, w, form, head_dim=None):
        shape = (*lead, width) if head_dim is None else (*lead[:2], width // head_dim, lead[2], head_dim)
        out = torch.full(shape, float("nan"), dtype=dtype, device=device)
        return region.small_product(a.contiguous().to(device), w.contiguous().to(device), out, rows, width, inner, form,
                                    1 if head_dim is None else lead[2], head_dim).cpu()

    got = product(g, weight, 0)
    assert bool(((got.double() - truth).abs() <= bound).all())
    heads = product(g, weight, 0, head_dim)
    assert torch.equal(heads, got.unflatten(-1, (-1, head_dim)).transpose(2, 3))
    assert bool(((product(g, weight.t(), 2).double() - truth).abs() <= bound).all())
    if rows % 8 == 0:
        assert bool(((product(g.reshape(rows, inner).t(), weight, 1).double() - truth).abs() <= bound).all())
    g[0, 0, 0, inner - 1], weight[inner - 1, width - 1] = float("inf"), float("inf")
    for got in (product(g, weight, 0), product(g, weight.t(), 2)):
        got = got.reshape(-1, width)
        assert bool(got[1:, :-1].isfinite().all()) and not bool(got[0].isfinite().any()) and not bool(got[:, -1].isfinite().any())


@pytest.mark.parametrize("height,width,rows", [(8, 8, 1), (72, 104, 17), (64, 136, 65), (256, 64, 384), (136, 72, 449), (520, 256, 1000)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_small_product_of_a_weight_gradient(height, width, rows, dtype, device):
    """Any number of rows; the bound of the test above."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    gen = torch.Generator().manual_seed(rows)
    g, x = torch.randn(rows, height, generator=gen).to(dtype), torch.randn(rows, width, generator=gen).to(dtype)
    got = region.small_product(g.to(device), x.to(device), torch.empty(height, width, dtype=dtype, device=device), height, width,
                               rows, 1).cpu()
    truth, sums = g.double().t() @ x.double(), g.double().abs().t() @ x.double().abs()
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = (rows + 1) * 2.0 ** -24 * sums * (1 + half_ulp) + half_ulp * truth.abs() + 2.0 ** -25
    assert bool(((got.double() - truth).abs() <= bound).all())


# uncut with tiles that the results end in, cut into two to many ranges (the last one short, or of a single step), results narrower than a
# tile; the first is one for the kernel above
@pytest.mark.parametrize("height,width,rows", [(136, 72, 449), (4104, 520, 700), (768, 3080, 1801), (264, 520, 2991), (8, 8, 8200), (136, 8, 4097),
                                               (64, 256, 20000), (1536, 520, 6000)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_weight_gradient_cut_into_ranges(height, width, rows, dtype, device):
    """The bound of the test above; a row past the end or of the next range in a sum would show in what is exact for small whole numbers; a
    value that is not finite stays in its row and column of the results."""
    from latent_bounded_interfaces_amd.hip.transformer import region

    gen = torch.Generator(device=device).manual_seed(rows)
    g, x = (torch.randn(rows, n, generator=gen, device=device).to(dtype) for n in (height, width))
    got = region.weight_gradient(g, x)
    assert torch.equal(got, region.weight_gradient(g, x))
    truth, sums = g.double().t().contiguous() @ x.double(), g.double().abs().t().contiguous() @ x.double().abs()
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = (rows + 1) * 2.0 ** -24 * sums * (1 + half_ulp) + half_ulp * truth.abs() + 2.0 ** -25
    assert bool(((got.double() - truth).abs() <= bound).all())
    g, x = (torch.randint(-1, 2, (rows, n), generator=gen, device=device).to(dtype) for n in (height, width))
    assert torch.equal(region.weight_gradient(g, x), (g.double().t().contiguous() @ x.double()).to(dtype))
    g[rows - 1, 3], x[rows // 2, 5] = float("inf"), float("nan")
    got = region.weight_gradient(g, x)
    got[3], got[:, 5] = 0, 0
    assert bool(got.isfinite().all())


def _small_block(dtype, device, *, dim=64, heads=2, kv=1, hd=32, hidden=96, layers=2, b=2, t=40, **more):
    backend = oreg.make_backend(dim=dim, n_heads=heads, n_kv_heads=kv, head_dim=hd, hidden=hidden, layers=layers, d_conv=4, dtype=dtype,
                                seed=7, **more).to(device)
    gen = torch.Generator().manual_seed(8)
    with torch.no_grad():
        _, cache = backend.forward_region(region_input=torch.randn(b, t, dim, generator=gen).to(dtype).to(device), region_index=0)
    return backend, cache, gen


def _launch_by_launch(monkeypatch, call):
    from latent_bounded_interfaces_amd.hip.transformer import region

    taken = []
    native = region._native_layer
    with monkeypatch.context() as patch:
        patch.setattr(region, "_native_layer", lambda *a: taken.append(native(*a)) or taken[-1])
        got = call()
    with monkeypatch.context() as patch:
        patch.setattr(region, "_native_layer", lambda *a: None)
        return got, call(), [one is not None for one in taken]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sizes", [dict(), dict(hd=64, t=64), dict(hd=64, heads=3, kv=3, t=300), dict(hd=128, t=130, rope_interleaved=True),
                                   dict(hd=40, dim=80, t=129, softmax_scale=0.2, residual_in_fp32=False), dict(t=1, b=1, layers=1)])
def test_native_layer_equals_its_launches(sizes, dtype, device, monkeypatch):
    """One call per block, and the same launches one by one: the same bits; dense and position-constant bases, parameter gradients."""
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    backend, cache, gen = _small_block(dtype, device, **sizes)
    lowering = HipTransformerLowering()
    b, t, dim = cache.region_input.shape
    basis = torch.randn(b, 3, t, dim, generator=gen).to(device)
    for cotangent in (basis, basis[:, :, :1].expand(b, 3, t, dim), basis.to(dtype)):
        keep = cotangent.clone()
        got, want, taken = _launch_by_launch(monkeypatch, lambda: lowering.input_pullback_basis(
            backend=backend, cache=cache, output_cotangent_basis=cotangent))
        assert all(taken) and torch.equal(got, want) and torch.equal(cotangent, keep)
    got, want, taken = _launch_by_launch(monkeypatch, lambda: lowering.parameter_vjp_with_input_cotangent(
        backend=backend, cache=cache, output_cotangent=basis[:, 0]))
    assert all(taken) and torch.equal(got[1], want[1]) and got[0].keys() == want[0].keys()
    for name, grad in want[0].items():
        assert torch.equal(got[0][name], grad) and got[0][name].dtype == grad.dtype, name


def _widened(node):
    """The same values in fp32, all the way down."""
    for name, value in vars(node).items():
        if torch.is_tensor(value) and value.is_floating_point():
            setattr(node, name, value.float())
        elif isinstance(value, list):
            for one in value:
                _widened(one)
        elif hasattr(value, "__dict__") and not torch.is_tensor(value):
            _widened(value)


# products of one to three times a small product's size, which the launches one by one leave to the library
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,b,t,p", [(512, 2, 65, 9), (768, 1, 258, 1), (512, 2, 512, 1)])
def test_native_layer_of_products_past_the_small_ones(dim, b, t, p, dtype, device, monkeypatch):
    """The two ways round differ in the order of fp32 sums: both are as far from fp32 arithmetic on the same values (a tenth of the error for
    what rounding does by chance, a quarter in gradients of a few hundred values)."""
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering
    from latent_bounded_interfaces_amd.hip.transformer import region

    backend, cache, gen = _small_block(dtype, device, dim=dim, heads=dim // 64, kv=dim // 64, hd=64, hidden=4 * dim, layers=1, b=b, t=t)
    work, grads = b * t * p * dim * 8 * dim / region._SMALL_PRODUCT, 8 * dim * dim / region._SMALL_PRODUCT_RESULTS  # the largest product and gradient
    assert 1 < max(work, grads) <= region._NATIVE_TIMES
    lowering = HipTransformerLowering()
    basis = torch.randn(b, p, t, dim, generator=gen).to(device)

    def pullback():
        return {"input": lowering.input_pullback_basis(backend=backend, cache=cache, output_cotangent_basis=basis)}

    def vjp():
        return lowering.parameter_vjp(backend=backend, cache=cache, output_cotangent=basis[:, 0])

    call = vjp if p == 1 else pullback
    got, want, taken = _launch_by_launch(monkeypatch, call)
    assert taken == [True] and got.keys() == want.keys()
    backend.float()
    _widened(cache)
    for name, truth in call().items():
        truth = truth.double()
        errors = [float((one[name].double() - truth).norm() / truth.norm()) for one in (got, want)]
        assert errors[0] <= (1.1 if truth.dim() > 1 else 1.25) * errors[1], (name, errors)
        assert errors[0] <= (2e-3 if dtype == torch.float16 else 1.5e-2), (name, errors)


def test_native_layer_leaves_what_it_does_not_take(device, monkeypatch):
    from latent_bounded_interfaces_amd.backends import HipTransformerLowering

    lowering = HipTransformerLowering()
    for dtype, sizes, expect in ((torch.float32, dict(), False), (torch.bfloat16, dict(bias=True), True), (torch.bfloat16, dict(hd=36, dim=72), False)):
        backend, cache, gen = _small_block(dtype, device, **sizes)
        b, t, dim = cache.region_input.shape
        basis = torch.randn(b, 2, t, dim, generator=gen).to(device)
        got, want, taken = _launch_by_launch(monkeypatch, lambda: lowering.input_pullback_basis(
            backend=backend, cache=cache, output_cotangent_basis=basis))
        assert torch.equal(got, want) and all(one is expect for one in taken)   # (biases take no part in the input pullback)
        got, want, taken = _launch_by_launch(monkeypatch, lambda: lowering.parameter_vjp(
            backend=backend, cache=cache, output_cotangent=basis[:, 0]))
        assert not any(taken) and all(torch.equal(got[name], grad) for name, grad in want.items())
    # weights off the 16-byte grid, and a cache that is not contiguous
    backend, cache, gen = _small_block(torch.bfloat16, device)
    block = backend.backbone.blocks[0]
    room = torch.empty(block.mlp.fc1.weight.numel() + 1, device=device, dtype=torch.bfloat16)
    moved = room[1:].view_as(block.mlp.fc1.weight)
    moved.copy_(block.mlp.fc1.weight.detach())
    block.mlp.fc1.weight.data = moved
    cache.layer_caches[1].attention.q_rope = cache.layer_caches[1].attention.q_rope.transpose(1, 2).contiguous().transpose(1, 2)
    b, t, dim = cache.region_input.shape
    basis = torch.randn(b, 2, t, dim, generator=gen).to(device)
    got, want, taken = _launch_by_launch(monkeypatch, lambda: lowering.input_pullback_basis(
        backend=backend, cache=cache, output_cotangent_basis=basis))
    assert taken == [True, False] and torch.equal(got, want)

