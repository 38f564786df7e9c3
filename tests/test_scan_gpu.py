"""Parity of the HIP suffix scan against the CPU oracle, through the C ABI (needs the GPU)."""
from __future__ import annotations

import json
from pathlib import Path

import pytest
import torch

from oracle import scan as oscan

pytestmark = pytest.mark.gpu

GOLDEN = json.loads((Path(__file__).parent / "golden" / "scan_known_answers.json").read_text())

# Every shape of the reference's tests (tests/test_interface_scan.py:45-53 and :78-86)
# plus ragged / non-power-of-two cases and each MFMA width with K not a power of two.
SHAPES = [
    (1, 0, 1), (1, 1, 1), (1, 1, 4), (2, 3, 5), (2, 4, 8), (4, 8, 16), (1, 16, 64),
    (1, 2, 16), (2, 4, 32), (2, 8, 64), (1, 16, 128), (1, 8, 256),
    (4, 8, 32), (3, 5, 32), (9, 7, 64), (5, 3, 128), (3, 5, 256), (2, 6, 48), (2, 3, 33), (1, 4, 100),
    (1, 3, 300), (2, 3, 512), (1, 2, 384),  # the widest matrix-core kernel, directly and through padding
    (1, 2, 520), (2, 5, 12),  # widths the scalar kernel still runs: past the largest matrix-core width, and tiny
    (17, 2, 256), (1, 1, 256), (2, 0, 32),
    (24, 14, 256), (33, 3, 256),  # d=256: 32-wide column blocks up to 32 batch elements, 64-wide beyond
]


# bf16 storage at d=256 runs on the 16-bit matrix cores.  By default the running suffix enters the products rounded to
# 16 significand bits (two bf16 planes): error against fp64 a hundred times inside the 2e-2 asked of 16-bit storage.
# exact_suffix=True (LBI_SCAN_EXACT_SUFFIX) keeps the fp32 value (three planes) and meets the fp32 bar.
BF16_D256_BAR = 2e-4
BF16_D256_EXACT_BAR = 1e-5


def _rel_err(actual: torch.Tensor, truth: torch.Tensor) -> float:
    """max over suffix matrices of max|diff| / max|truth| (fp64 truth)."""
    diff = (actual.double() - truth).abs().flatten(2).max(dim=2).values
    ref = truth.abs().flatten(2).max(dim=2).values.clamp_min(1e-30)
    return float((diff / ref).max())


def _scan(mats_cpu: torch.Tensor, device) -> torch.Tensor:
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks

    mats = mats_cpu.to(device)
    keep = mats.clone()
    out = suffix_scan_pullbacks(mats)
    torch.cuda.synchronize()
    assert torch.equal(mats, keep), "input was modified"
    return out.cpu()


def test_known_answer_2x2(device):
    case = GOLDEN["order_case_2x2"]
    out = _scan(torch.tensor(case["mats"], dtype=torch.float32), device)
    assert torch.equal(out, torch.tensor(case["suffix"], dtype=torch.float32))


@pytest.mark.parametrize("shape", SHAPES)
def test_fp32_matches_oracle(shape, device):
    bsz, count, rank = shape
    mats, _ = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=0)
    out = _scan(mats, device)
    assert out.shape == (bsz, count + 1, rank, rank)
    assert out.dtype == torch.float32
    assert torch.equal(out[:, count], torch.eye(rank).expand(bsz, rank, rank))
    truth = oscan.suffix_scan_sequential(mats, dtype=torch.float64)
    assert _rel_err(out, truth) <= 1e-5  # bar for the fp32 scan
    # The reference's CPU algorithm (log-depth order) agrees to the same bar.
    levels = oscan.suffix_scan_levels(mats)
    assert _rel_err(out, levels.double()) <= 1e-5
    # Sequential fp32 product has the SAME association order as the kernel.
    seq = oscan.suffix_scan_sequential(mats)
    assert torch.allclose(out, seq, atol=2e-5, rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 8, 64), (2, 5, 256), (3, 4, 24), (2, 6, 128), (2, 9, 32)])
def test_low_precision_storage_promotes_to_fp32(shape, dtype, device):
    # reference tests/test_interface_scan.py:104-115
    bsz, count, rank = shape
    mats, _ = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=0)
    mats = mats.to(dtype)
    out = _scan(mats, device)
    assert out.dtype == torch.float32
    truth = oscan.suffix_scan_sequential(mats.float(), dtype=torch.float64)
    # Inputs are rounded before both sides see them, so only fp32 accumulation differs.
    bar = BF16_D256_BAR if (dtype == torch.bfloat16 and rank == 256) else 1e-5
    assert _rel_err(out, truth) <= bar
    assert torch.allclose(out, oscan.suffix_scan_sequential(mats.float()), atol=2e-1, rtol=5e-3)
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks

    exact = suffix_scan_pullbacks(mats.to(device), exact_suffix=True).cpu()
    assert _rel_err(exact, truth) <= 1e-5


def test_permutations_are_exact(device):
    gen = torch.Generator().manual_seed(5)
    rank, count = 64, 9
    perms = [torch.randperm(rank, generator=gen) for _ in range(count)]
    mats = torch.stack([torch.eye(rank)[p] for p in perms]).unsqueeze(0).repeat(3, 1, 1, 1)
    out = _scan(mats, device)
    idx = torch.arange(rank)
    for r in range(count - 1, -1, -1):
        idx = idx[perms[r]]
        assert torch.equal(out[1, r], torch.eye(rank)[idx])


@pytest.mark.parametrize("shape", [(1, 0, 3), (2, 1, 8), (3, 5, 7), (4, 8, 32), (2, 6, 64), (3, 9, 128),
                                   (5, 12, 256), (2, 3, 100), (2, 4, 260), (2, 0, 256), (3, 1, 256), (1, 2, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_cotangent_chain_matches_oracle(shape, dtype, device):
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents

    bsz, count, rank = shape
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=1)
    mats = mats.to(dtype)
    out = suffix_scan_cotangents(mats.to(device), g.to(device)).cpu()
    assert out.shape == (bsz, count + 1, rank) and out.dtype == torch.float32
    assert torch.equal(out[:, count], g)
    truth = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    scale = truth.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((out.double() - truth).abs() / scale).max()) <= 1e-5
    case = GOLDEN["order_case_2x2"]
    got = suffix_scan_cotangents(torch.tensor(case["mats"]).to(device), torch.tensor(case["g"]).to(device))
    assert torch.equal(got.cpu(), torch.tensor(case["cotangents"]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [65, 95, 96, 129, 160, 161, 191, 192, 193])
@pytest.mark.parametrize("bsz,count", [(1, 1), (2, 2), (1, 40), (3, 13), (45, 14)])
def test_widths_between_powers_of_two(rank, bsz, count, dtype, device):
    """Both forms of the scan (one chain; chunks side by side) at 96, 160 and 192 columns and what is padded to them,
    on tensors that start off the 16-byte grid too."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks, suffix_scan_pullbacks_and_cotangents

    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=rank + count)
    mats = mats.to(dtype).to(device)
    off = torch.empty(mats.numel() + 1, dtype=dtype, device=device)[1:].view(mats.shape).copy_(mats)
    g_off = torch.empty(g.numel() + 1, device=device)[1:].view(g.shape).copy_(g)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats, g.to(device))
    out_off, cot_off = suffix_scan_pullbacks_and_cotangents(off, g_off)
    assert torch.equal(out, out_off) and torch.equal(cot, cot_off)
    only = suffix_scan_pullbacks(mats)
    truth = oscan.suffix_scan_sequential(mats.cpu(), dtype=torch.float64)
    want = oscan.suffix_cotangents_sequential(mats.cpu().double(), g.double())
    bar = 2e-4 if dtype == torch.bfloat16 and rank > 192 else 1e-5   # bf16 at 193: the width-256 kernel's two planes
    for result in (out, only):
        result = result.cpu()
        err = (result.double() - truth).abs().flatten(2).amax(2) / truth.abs().flatten(2).amax(2)
        assert float(err.max()) <= bar
        assert torch.equal(result[:, count], torch.eye(rank).expand(bsz, -1, -1))
    scale = want.abs().amax(dim=-1, keepdim=True)
    assert float(((cot.cpu().double() - want).abs() / scale).max()) <= max(bar, 3e-5)   # products applied to g


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [17, 31, 33, 63, 97, 127, 131, 254])
@pytest.mark.parametrize("bsz,count", [(1, 1), (2, 3), (1, 40), (520, 3)])
def test_widths_read_where_they_lie(rank, bsz, count, dtype, device):
    """Widths between the kernels' own, on tensors that start off the grid too; an infinity that begins a row stays out of
    the row before, whose last chunk reads past its end."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks, suffix_scan_pullbacks_and_cotangents

    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=rank + count)
    mats = mats.to(dtype)
    truth = oscan.suffix_scan_sequential(mats, dtype=torch.float64)
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    dev = torch.empty(mats.numel() + 1, dtype=dtype, device=device)[1:].view(mats.shape).copy_(mats)
    out, cot = suffix_scan_pullbacks_and_cotangents(dev, g.to(device))
    only = suffix_scan_pullbacks(mats.to(device))
    bar = 2e-4 if dtype == torch.bfloat16 and rank > 192 else 1e-5   # the width-256 kernel's two planes
    for result in (out.cpu(), only.cpu()):
        err = (result.double() - truth).abs().flatten(2).amax(2) / truth.abs().flatten(2).amax(2)
        assert float(err.max()) <= bar
    scale = want.abs().amax(dim=-1, keepdim=True)
    assert float(((cot.cpu().double() - want).abs() / scale).max()) <= max(bar, 3e-5)   # products applied to g
    if 1 < count < 12:
        mats[-1, 0, 9, 0] = float("inf")
        out, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
        for result in (out[-1, 0], cot[-1, 0]):
            bad = ~result.isfinite()
            assert bool(bad[9].all()) and int(bad.sum()) == bad[9].numel()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [130, 192, 256])
@pytest.mark.parametrize("bsz,count", [(1, 40), (2, 5), (40, 4)])
@pytest.mark.parametrize("kind", ["inf", "nan", "huge", "tiny", "zero_rows"])
def test_values_outside_the_range_of_the_planes(kind, rank, bsz, count, dtype, device):
    """Above 128 columns an fp32 number is the sum of three bf16 ones; what they cannot hold (infinities, values next to
    the largest, products far below 1) comes out as fp32 arithmetic gives it, and stays where it belongs."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks, suffix_scan_pullbacks_and_cotangents

    if dtype == torch.bfloat16 and rank == 256 and (bsz, count) != (1, 40):
        pytest.skip("two planes without a check: the width-256 bf16 kernels")
    if kind in ("inf", "nan") and bsz == 1:
        pytest.skip("chunks side by side: infinities cancel in another order than along one chain")
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=rank + count)
    at = (bsz - 1, count // 2)
    if kind == "inf":
        mats[at][3, rank - 2] = float("inf")
    elif kind == "nan":
        mats[at][rank - 1, 0] = float("nan")
    elif kind == "huge":   # the largest finite value, which rounds to infinity in bf16, through identities
        mats[:] = torch.eye(rank)
        mats[at][5, rank - 1] = torch.finfo(dtype).max
        g *= 0.1 / g.abs().max()
    elif kind == "tiny":   # down to 2^-120 over the chain, and one block of rows only
        mats[at[0]] *= 2.0 ** (-120.0 / count)
        mats[0, count - 1, 32:64] *= 2.0 ** -12
    else:
        mats[at][40:80] = 0.0
    mats = mats.to(dtype)
    truth = oscan.suffix_scan_sequential(mats.float(), dtype=torch.float64)
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    out, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
    assert torch.equal(torch.nan_to_num(out), torch.nan_to_num(suffix_scan_pullbacks(mats.to(device)))) or bsz == 40
    for got, ref in ((out.cpu().double(), truth), (cot.cpu().double()[:, :, None], want[:, :, None])):
        assert torch.equal(got.isnan(), ref.isnan())
        ok = ref.isfinite()
        assert torch.equal(got[~ok & ~ref.isnan()], ref[~ok & ~ref.isnan()])
        scale = torch.where(ok, ref.abs(), 0.0).amax(-1, keepdim=True).clamp_min(1e-37)   # of every row
        assert float((torch.where(ok, (got - ref).abs(), 0.0) / scale).max()) <= 5e-5     # 40 roundings a row, ~1e-5 seen


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [160, 192, 256])
@pytest.mark.parametrize("at", [(3, 5), (37, 40), (158, 150), (3, 100)])
@pytest.mark.parametrize("value", ["inf", "max"])
def test_fused_chain_meets_what_planes_cannot_hold(value, at, rank, dtype, device):
    """An infinity and the largest finite value, in the columns that a wave's first product step takes (its own rows') and in
    another: the cotangents come out as fp32 arithmetic gives them."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents

    if dtype == torch.bfloat16 and rank == 256:
        pytest.skip("two planes without a check: the width-256 bf16 kernels")
    gen = torch.Generator().manual_seed(rank)
    mats = torch.eye(rank, dtype=dtype).repeat(3, 9, 1, 1)
    mats[1, 2][at] = torch.finfo(dtype).max if value == "max" else float("inf")
    g = torch.rand(3, rank, generator=gen) * 0.1 + 0.01
    _, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    got = cot.cpu().double()
    assert torch.equal(got.isnan(), want.isnan())
    ok = want.isfinite()
    assert torch.equal(got[~ok & ~want.isnan()], want[~ok & ~want.isnan()])
    # a row has two terms: three roundings of 2^-24
    assert float(((got - want).abs()[ok] / want.abs()[ok]).max()) <= 2e-7


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rank", [140, 192, 256])
@pytest.mark.parametrize("bsz,count", [(3, 5), (20, 14), (1, 40)])
@pytest.mark.parametrize("kind", ["column", "row", "matrix", "subnormal", "large"])
def test_tiny_numbers_keep_their_accuracy(kind, rank, bsz, count, dtype, device):
    """Numbers whose lower planes would fall below the smallest that bf16 holds: one column of the products, one row of a
    matrix, a whole small matrix times a large suffix; and products past the other end, back in range a step later.  The
    error is that of the tiny numbers' own row or column."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks, suffix_scan_pullbacks_and_cotangents

    if dtype == torch.bfloat16 and rank == 256 and (bsz, count) != (1, 40):
        pytest.skip("two planes: the width-256 bf16 kernels")
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=rank + count)
    if kind == "column":
        mats[:, count - 1, :, 7] *= 2.0 ** -115
    elif kind == "row":
        mats[:, 1, 9] *= 2.0 ** -115
    else:
        mats[:, 1] *= {"matrix": 2.0 ** -118, "subnormal": 2.0 ** -126, "large": 2.0 ** -90}[kind]
        mats[:, 2] *= 2.0 ** (90 if kind == "large" else 60)
    mats = mats.to(dtype)
    truth = oscan.suffix_scan_sequential(mats.float(), dtype=torch.float64)
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    out, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
    along = 2 if kind == "column" else 3
    for got in (out, suffix_scan_pullbacks(mats.to(device))):
        err = (got.cpu().double() - truth).abs().amax(along) / truth.abs().amax(along).clamp_min(1e-300)
        assert float(err.max()) <= 1e-5
    # entry by entry against the sizes of its terms, those of the chain or those of the finished product
    size = torch.maximum(torch.einsum("bkij,bkj->bki", mats.double().abs(), want[:, 1:].abs()),
                         torch.einsum("bkij,bj->bki", truth[:, :count].abs(), g.double().abs()))
    assert float(((cot.cpu().double() - want).abs()[:, :count] / size).max()) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 40, 200), (1, 40, 131), (2, 33, 170), (1, 100, 253), (1, 13, 129), (1, 70, 45)])
def test_chunked_scan_takes_nothing_from_the_result_buffer(shape, dtype, device):
    """The chunk totals are parked in result slots: what lay in the buffer before, NaN and the largest numbers included, leaves
    no trace, at widths whose rows end inside a tile."""
    from latent_bounded_interfaces_amd import _lib

    bsz, count, rank = shape
    if dtype != torch.float32 and rank > 128 and rank % 2:
        pytest.skip("odd 16-bit widths run on padded copies")
    mats = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=3)[0].to(dtype)
    truth = oscan.suffix_scan_sequential(mats.float(), dtype=torch.float64)
    mats = mats.to(device)
    results = []
    for fill in (0.0, float("nan"), torch.finfo(torch.float32).max):
        out = torch.full((bsz, count + 1, rank, rank), fill, device=device)
        with _lib.device_guard(mats.device):
            _lib.check(_lib.load().lbi_suffix_scan_ex(mats.data_ptr(), None, out.data_ptr(), None, bsz, count, rank,
                                                      _lib.dtype_code(dtype), _lib.LBI_F32, 0,
                                                      _lib.current_stream_ptr(mats.device)), "lbi_suffix_scan_ex")
        results.append(out)
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])
    assert _rel_err(results[0].cpu(), truth) <= 1e-5


# widths of one to eight row tiles, whole and not, in whole 16-byte pieces or not, either side of the lines of the narrow chain; one matrix
# and chains that end anywhere in a trip of the rows' ring
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank,bsz,count", [(2, 1, 1), (7, 9, 13), (15, 3, 40), (16, 300, 2), (17, 8, 3), (33, 2, 19), (33, 2, 21), (48, 65, 6),
                                            (56, 4, 17), (64, 5, 31), (72, 3, 9), (80, 17, 14), (96, 2, 12), (112, 3, 7), (128, 9, 23), (120, 257, 2),
                                            (32, 1025, 3)])
def test_narrow_cotangent_chain(rank, bsz, count, dtype, device):
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents

    gen = torch.Generator(device=device).manual_seed(rank + count)
    mats = torch.randn(bsz, count, rank, rank, generator=gen, device=device) * (0.01 / rank) ** 0.5
    mats.diagonal(dim1=-2, dim2=-1).add_(1.0)
    mats, g = mats.to(dtype), torch.randn(bsz, rank, generator=gen, device=device)
    got = suffix_scan_cotangents(mats, g)
    v, want = g.double(), [g.double()]
    for r in range(count - 1, -1, -1):
        v = (mats[:, r].double() @ v.unsqueeze(-1)).squeeze(-1)
        want.append(v)
    want = torch.stack(want[::-1], dim=1)
    # each step rounds each of its rank terms and sums once, of terms whose absolute values sum to at most twice the result's norm
    bound = 2 * count * (rank + 8) * 2.0 ** -24 * float(want.norm(dim=-1).max())
    assert got.shape == want.shape and float((got.double() - want).abs().max()) <= bound
    at = count // 2
    mats[bsz - 1, at, rank - 1, 0] = float("inf")
    again = suffix_scan_cotangents(mats, g)
    finite = again.isfinite()
    assert bool(finite[:bsz - 1].all()) and bool(finite[bsz - 1, at + 1:].all()) and bool(finite[bsz - 1, at, :rank - 1].all())
    assert not bool(finite[bsz - 1, at, rank - 1]) and torch.equal(again[:bsz - 1], got[:bsz - 1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [17, 63, 65, 127, 129, 191, 193, 198, 254, 255])
@pytest.mark.parametrize("bsz,count", [(1, 1), (3, 9)])
def test_cotangent_chain_rows_in_registers(rank, bsz, count, dtype, device):
    """Widths up to 256 whose rows are no whole 16-byte pieces: edges of the 64-column blocks a lane holds."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents

    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=rank)
    mats = mats.to(dtype)
    mats[0, 0, 0, rank - 1] = float("inf")   # reaches the one entry that multiplies it, from the row's last column
    out = suffix_scan_cotangents(mats.to(device), g.to(device)).cpu()
    truth = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    assert torch.equal(out[:, count], g)
    finite = torch.isfinite(truth)
    assert torch.equal(torch.isinf(out), torch.isinf(truth)) and not torch.isnan(out).any()
    scale = truth.where(finite, torch.zeros(())).abs().amax(dim=-1, keepdim=True).clamp_min(1e-30)
    assert float(((out.double() - truth).abs() / scale)[finite].max()) <= 1e-5


@pytest.mark.parametrize("dtype,rank", [(torch.float32, 184), (torch.float32, 252), (torch.bfloat16, 132), (torch.float16, 204)])
@pytest.mark.parametrize("bsz", [3, 1023, 1024])
def test_cotangent_chain_rows_of_many_chains(bsz, dtype, rank, device):
    """Rows of whole 4-element pieces: in registers for few chains, one at a time from four chains per CU on (256 CUs)."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents

    gen = torch.Generator(device=device).manual_seed(rank)
    mats = (torch.randn(bsz, 3, rank, rank, generator=gen, device=device) * rank ** -0.5).to(dtype)
    g = torch.randn(bsz, rank, generator=gen, device=device)
    out = suffix_scan_cotangents(mats, g)
    assert torch.equal(out[:, 3], g)
    want = g.double()
    for r in (2, 1, 0):
        want = torch.bmm(mats[:, r].double(), want.unsqueeze(-1)).squeeze(-1)
        err = (out[:, r].double() - want).abs().amax() / want.abs().amax()
        assert float(err) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bsz,count", [(1, 2), (3, 5), (13, 128), (64, 128), (64, 9), (65, 11)])
def test_cotangent_chain_on_four_workgroups_per_element(bsz, count, dtype, device):
    """d = 256 with at most a quarter as many chains as CUs: four workgroups share a chain and exchange each step's
    vector through the result array (marker words).  Against the fp64 chain, terminal cotangent in place, no marker
    left behind, reruns bit-identical; 65 chains take the one-workgroup kernel and must agree to rounding."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents

    mats, g = oscan.make_scan_inputs(bsz, count, 256, kind="near_identity", seed=21)
    mats_d, g_d = mats.to(device).to(dtype), g.to(device)
    out = suffix_scan_cotangents(mats_d, g_d)
    assert torch.equal(out, suffix_scan_cotangents(mats_d, g_d)), "reruns differ"
    assert bool(torch.isfinite(out).all()) and torch.equal(out[:, count], g_d)
    truth = oscan.suffix_cotangents_sequential(mats_d.double().cpu(), g.double())
    scale = truth.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((out.cpu().double() - truth).abs() / scale).max()) <= 1e-5


def test_cotangent_chain_partner_timeout_path_in_subprocess(device):
    """A reader that gives up on its partners (forced from the host: LBI_COT_SPIN_LIMIT=0, no poll ever succeeds in
    time) forms every missing entry itself: every wave still reaches every barrier and the chain is still right, in
    the cotangent-only kernel and in the chain waves of the fused bf16 scan."""
    import os
    import subprocess
    import sys

    code = (
        "import torch, sys; sys.path.insert(0, %r);"
        "from oracle import scan as o;"
        "from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents as f;"
        "worst = 0.0\n"
        "from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents as fused\n"
        "for dt in (torch.float32, torch.bfloat16):\n"
        "    m, g = o.make_scan_inputs(5, 23, 256, kind='near_identity', seed=3); m = m.to(dt)\n"
        "    out = f(m.cuda(), g.cuda()).cpu().double()\n"
        "    t = o.suffix_cotangents_sequential(m.double(), g.double())\n"
        "    worst = max(worst, float(((out - t).abs() / t.abs().amax(2, keepdim=True)).max()))\n"
        "m, g = o.make_scan_inputs(20, 7, 256, kind='near_identity', seed=4); m = m.to(torch.bfloat16)\n"
        "mats, cot = fused(m.cuda(), g.cuda())\n"
        "t = o.suffix_cotangents_sequential(m.double(), g.double())\n"
        "worst = max(worst, float(((cot.cpu().double() - t).abs() / t.abs().amax(2, keepdim=True)).max()))\n"
        "tm = o.suffix_scan_sequential(m.float(), dtype=torch.float64)\n"
        "assert float(((mats.cpu().double() - tm).abs().flatten(2).amax(2) / tm.abs().flatten(2).amax(2)).max()) <= 2e-4\n"
        "print(worst); sys.exit(0 if worst <= 1e-5 else 1)"
    ) % str(Path(__file__).resolve().parents[1])
    env = dict(os.environ, LBI_COT_SPIN_LIMIT="0")
    res = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stdout + res.stderr


@pytest.mark.parametrize("shape", [(1, 0, 3), (2, 1, 8), (3, 5, 7), (4, 8, 32), (2, 6, 64), (3, 9, 128), (5, 12, 256),
                                   (9, 1, 256), (2, 2, 32), (2, 3, 100), (1, 1, 64), (2, 3, 512), (1, 2, 300)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_fused_scan_and_cotangents(shape, dtype, device):
    """One pass giving both results equals the two separate entry points (bit-exact for the
    matrices) and the oracle for the cotangents."""
    from latent_bounded_interfaces_amd.hip.interface import (
        suffix_scan_pullbacks,
        suffix_scan_pullbacks_and_cotangents,
    )

    bsz, count, rank = shape
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=4)
    mats = mats.to(dtype)
    mats_d, g_d = mats.to(device), g.to(device)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats_d, g_d)
    assert torch.equal(out, suffix_scan_pullbacks(mats_d))
    assert cot.shape == (bsz, count + 1, rank) and cot.dtype == torch.float32
    assert torch.equal(cot[:, count].cpu(), g)
    truth = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    scale = truth.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((cot.cpu().double() - truth).abs() / scale).max()) <= 1e-5


@pytest.mark.parametrize("shape", [(2, 5, 256), (9, 1, 256), (3, 12, 256), (2, 6, 64), (17, 9, 256), (64, 3, 256),
                                   (65, 3, 256)])
def test_fused_scan_and_cotangents_bf16_storage(shape, device):
    """bf16 storage at d=256: the matrices-only entry runs the column-owner kernel; the fused entry the same kernel
    with chain waves (up to 64 batch elements: the four workgroups of an element exchange the chain vector) or the
    row-owner split kernel (larger batches); with ``exact_suffix`` both are exact-split fp32 products in different
    summation orders, by default the suffix operand is rounded to 16 significand bits in both."""
    from latent_bounded_interfaces_amd.hip.interface import (
        suffix_scan_pullbacks,
        suffix_scan_pullbacks_and_cotangents,
    )

    bsz, count, rank = shape
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=6)
    mats = mats.to(torch.bfloat16)
    mats_d, g_d = mats.to(device), g.to(device)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats_d, g_d)
    truth = oscan.suffix_scan_sequential(mats.float(), dtype=torch.float64)
    bar = BF16_D256_BAR if rank == 256 else 1e-5
    assert _rel_err(out.cpu(), truth) <= bar
    assert _rel_err(suffix_scan_pullbacks(mats_d).cpu(), truth) <= bar
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    scale = want.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((cot.cpu().double() - want).abs() / scale).max()) <= 1e-5  # the chain itself is fp32 throughout
    out3, cot3 = suffix_scan_pullbacks_and_cotangents(mats_d, g_d, exact_suffix=True)
    assert _rel_err(out3.cpu(), truth) <= BF16_D256_EXACT_BAR
    assert _rel_err(suffix_scan_pullbacks(mats_d, exact_suffix=True).cpu(), truth) <= BF16_D256_EXACT_BAR
    assert torch.equal(cot3, cot)
    if shape == (2, 5, 256):                   # (short chains of few elements; long ones run the fp32 chunked form)
        assert not torch.equal(out3, out)      # the flag does select another kernel instantiation


def test_benchmark_shape_properties(device):
    """B=64, K=128, d=256: size-independent checks (recurrence, identity tail, reruns bit-stable)."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents, suffix_scan_pullbacks

    bsz, count, rank = 64, 128, 256
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="near_identity", seed=0)
    mats_d = mats.to(device)
    out = suffix_scan_pullbacks(mats_d)
    again = suffix_scan_pullbacks(mats_d)
    assert torch.equal(out, again), "reruns differ"
    assert torch.equal(out[:, count], torch.eye(rank, device=device).expand(bsz, rank, rank))
    # out[r] == mats[r] @ out[r+1] for a sample of r, checked in fp64 on the device.
    for r in (0, 1, 63, 126, 127):
        want = torch.matmul(mats_d[:, r].double(), out[:, r + 1].double())
        err = (out[:, r].double() - want).abs().amax() / want.abs().amax()
        assert float(err) <= 2e-6, (r, float(err))
    # Full fp64 truth for two batch elements on the CPU.
    pick = [0, 37]
    truth = oscan.suffix_scan_sequential(mats[pick], dtype=torch.float64)
    assert _rel_err(out[pick].cpu(), truth) <= 1e-5
    # Cotangents: chain == suffix matrices applied to g (the reference's interface_scan_rms check,
    # backward/scan.py:63-72, bar 1e-5 RMS).
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents

    g_d = g.to(device)
    chain = suffix_scan_cotangents(mats_d, g_d)
    via_mats = torch.einsum("bkij,bj->bki", out.double(), g_d.double())
    rms = float(torch.sqrt(((chain.double() - via_mats) ** 2).mean()))
    assert rms < 1e-5
    fused_out, fused_cot = suffix_scan_pullbacks_and_cotangents(mats_d, g_d)
    assert torch.equal(fused_out, out)
    assert float(torch.sqrt(((fused_cot.double() - via_mats) ** 2).mean())) < 1e-5
    # bf16 storage, fp32 accumulate: inputs are rounded to bf16 before either path sees
    # them; bar 2e-2 against the fp32 path on the same (rounded) inputs.
    mats_bf16 = mats_d.to(torch.bfloat16)
    out_bf16 = suffix_scan_pullbacks(mats_bf16)
    out_ref = suffix_scan_pullbacks(mats_bf16.float())
    rel = (out_bf16 - out_ref).abs().flatten(2).amax(dim=2) / out_ref.abs().flatten(2).amax(dim=2)
    assert float(rel.max()) <= 2e-2
    truth_bf = oscan.suffix_scan_sequential(mats_bf16[pick].float().cpu(), dtype=torch.float64)
    assert _rel_err(out_bf16[pick].cpu(), truth_bf) <= BF16_D256_BAR


@pytest.mark.parametrize("bsz", [1, 2, 4, 8])
@pytest.mark.parametrize("kind", ["near_identity", "randn"])
def test_k_parallel_scan_at_small_batches(bsz, kind, device):
    """K=128, d=256 with so few batch elements that the chain is cut into chunks that run side by side
    (three launches): same results as the sequential product to the fp32 bar, identity tail, cotangents,
    reruns bit-identical, fused entry == matrices-only entry."""
    from latent_bounded_interfaces_amd.hip.interface import (suffix_scan_pullbacks,
                                                             suffix_scan_pullbacks_and_cotangents)

    count, rank = 128, 256
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind=kind, seed=7)
    mats_d, g_d = mats.to(device), g.to(device)
    out = suffix_scan_pullbacks(mats_d)
    assert torch.equal(out, suffix_scan_pullbacks(mats_d)), "reruns differ"
    assert torch.equal(out[:, count], torch.eye(rank, device=device).expand(bsz, rank, rank))
    assert torch.equal(out[:, count - 1], mats_d[:, count - 1])
    truth = oscan.suffix_scan_sequential(mats, dtype=torch.float64)
    assert _rel_err(out.cpu(), truth) <= 1e-5
    fused, cot = suffix_scan_pullbacks_and_cotangents(mats_d, g_d)
    assert torch.equal(fused, out)
    assert torch.equal(cot[:, count].cpu(), g)
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    scale = want.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((cot.cpu().double() - want).abs() / scale).max()) <= 1e-5
    again = suffix_scan_pullbacks_and_cotangents(mats_d, g_d)
    assert torch.equal(again[0], fused) and torch.equal(again[1], cot)


# chains long enough to be cut, at every matrix-core width the chunked form runs, lengths that leave a ragged or
# one-matrix last chunk, batch sizes either side of the 8-chain launch mapping
K_PARALLEL_SHAPES = [(1, 13, 32), (1, 37, 64), (2, 100, 128), (3, 61, 256), (1, 12, 256), (1, 129, 256), (9, 33, 32),
                     (7, 50, 64), (2, 17, 100), (1, 40, 200),
                     # chunk boundaries sit at cL - 1: lengths that make the last chunk one matrix, a full chunk, and
                     # the shortest chains the planner cuts
                     (1, 15, 256), (1, 16, 256), (2, 47, 256), (1, 255, 128), (4, 128, 32), (1, 14, 64)]


@pytest.mark.parametrize("shape", K_PARALLEL_SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_k_parallel_scan_shapes(shape, dtype, device):
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents

    bsz, count, rank = shape
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="randn", seed=8)
    mats = mats.to(dtype)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
    truth = oscan.suffix_scan_sequential(mats.float(), dtype=torch.float64)
    assert torch.equal(out[:, count].cpu(), torch.eye(rank).expand(bsz, rank, rank))
    assert _rel_err(out.cpu(), truth) <= 1e-5
    # The chunks share no chain, so these cotangents are the finished products applied to g, which is how the
    # reference gets them (backward/suffix_scan.py:49-53): the 1e-5 of a product can be amplified where the
    # mat-vec cancels, hence 3e-5 per vector here, and the reference's own bar for this quantity, an RMS
    # difference to the sequential chain below 1e-5 (backward/scan.py:63-72, tests/test_lbi_gradient_parity.py:44).
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    scale = want.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((cot.cpu().double() - want).abs() / scale).max()) <= 3e-5
    assert float(torch.sqrt((((cot.cpu().double() - want) / scale) ** 2).mean())) <= 1e-5


@pytest.mark.parametrize("shape", [(1, 1000, 64), (1, 520, 256), (3, 300, 128)])
def test_k_parallel_scan_long_chains(shape, device):
    """Chains of hundreds of matrices (many chunks: five or six levels over the chunk totals) on the benchmark's
    near-identity inputs: every product against the fp64 sequential product, the identity tail, reruns bit for
    bit, and the fused cotangents against the fp64 chain."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks, suffix_scan_pullbacks_and_cotangents

    bsz, count, rank = shape
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="near_identity", seed=9)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
    truth = oscan.suffix_scan_sequential(mats, dtype=torch.float64)
    assert torch.equal(out[:, count].cpu(), torch.eye(rank).expand(bsz, rank, rank))
    assert _rel_err(out.cpu(), truth) <= 1e-5
    assert torch.equal(out, suffix_scan_pullbacks(mats.to(device)))
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    scale = want.abs().amax(dim=2, keepdim=True).clamp_min(1e-30)
    assert float(((cot.cpu().double() - want).abs() / scale).max()) <= 3e-5


@pytest.mark.parametrize("chunk,totals_chain", [(0, 0), (2, 0), (3, 0), (5, 0), (16, 0), (3, 1), (5, 1)])
def test_k_parallel_scan_forced_chunk_lengths_in_subprocess(chunk, totals_chain, device):
    """LBI_SCAN_CHUNK forces the chunk length (0: the plain chain): every cut of K=13 / 29 / 33 / 64, including a
    one-matrix last chunk, meets the bar, with and without the cotangent chain.  The products of the chunk totals
    are formed in log depth where there are eight chunks or more and chunks of three matrices or more (chunk
    lengths 3 and 5 at K = 33 / 64 here; length 3 uses the last free slot of a chunk), as one chain otherwise;
    LBI_SCAN_TOTALS_CHAIN=1 forces the chain."""
    import os
    import subprocess
    import sys

    code = (
        "import torch, sys; sys.path.insert(0, %r);"
        "from oracle import scan as o;"
        "from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks as s, "
        "suffix_scan_pullbacks_and_cotangents as f;"
        "worst = 0.0\n"
        "for shape in ((1, 13, 64), (2, 33, 256), (1, 64, 32), (3, 21, 128), (1, 29, 256)):\n"
        "    m, g = o.make_scan_inputs(*shape, kind='randn', seed=5)\n"
        "    t = o.suffix_scan_sequential(m, dtype=torch.float64)\n"
        "    c = o.suffix_cotangents_sequential(m.double(), g.double())\n"
        "    out, cot = f(m.cuda(), g.cuda())\n"
        "    assert torch.equal(out, s(m.cuda()))\n"
        "    worst = max(worst, float(((out.cpu().double() - t).abs().flatten(2).amax(2) / t.abs().flatten(2).amax(2)).max()))\n"
        "    worst = max(worst, float(((cot.cpu().double() - c).abs() / c.abs().amax(2, keepdim=True)).max()))\n"
        "print(worst); sys.exit(0 if 0.0 < worst <= 1e-5 else 1)"
    ) % str(Path(__file__).resolve().parents[1])
    env = dict(os.environ, LBI_SCAN_CHUNK=str(chunk), LBI_SCAN_TOTALS_CHAIN=str(totals_chain))
    res = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stdout + res.stderr


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 4, 5), (3, 6, 16), (2, 9, 64), (1, 3, 100), (2, 5, 256), (1, 2, 300)])
def test_suffix_apply_matches_einsum(shape, device):
    """``lbi_suffix_apply``: every matrix of a stack applied to its batch element's vector, in fp64 on the CPU."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_apply

    bsz, count, rank = shape
    gen = torch.Generator().manual_seed(rank)
    suffix = torch.randn(bsz, count, rank, rank, generator=gen)
    g = torch.randn(bsz, rank, generator=gen)
    got = suffix_apply(suffix.to(device), g.to(device)).cpu()
    want = torch.einsum("bkij,bj->bki", suffix.double(), g.double())
    assert got.shape == (bsz, count, rank) and got.dtype == torch.float32
    assert torch.allclose(got.double(), want, atol=1e-5 * float(want.abs().max()), rtol=1e-5)
    with pytest.raises(ValueError):
        suffix_apply(suffix.to(device), g[:, :-1].to(device)) if rank > 1 else suffix_apply(suffix[0].to(device), g.to(device))


def test_backward_module_contract(device):
    """Counterpart functions of reference backward/suffix_scan.py keep its edge cases."""
    from latent_bounded_interfaces_amd.backward import suffix_scan as bs

    mats, g = oscan.make_scan_inputs(3, 5, 16, kind="randn", seed=2)
    jts = [mats[:, r].to(device) for r in range(5)]
    g_d = g.to(device)
    suffix = bs.compose_suffix_jacobian_t(jts)
    assert len(suffix) == 6 and all(s.shape == (3, 16, 16) and s.is_contiguous() for s in suffix)
    truth = oscan.suffix_scan_sequential(mats, dtype=torch.float64)
    assert _rel_err(torch.stack([s.cpu() for s in suffix], 1), truth) <= 1e-5
    assert bs.compose_suffix_jacobian_t([]) == []
    with pytest.raises(ValueError):
        bs.compose_suffix_jacobian_t([torch.zeros(2, 3, 4, device=device)])
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    for flag in (False, True):
        got = bs.propagate_state_adjoint_with_jacobian_scan(jts, g_d, materialize_suffix=flag)
        assert len(got) == 6
        assert torch.allclose(torch.stack([x.cpu() for x in got], 1).double(), want, atol=1e-5, rtol=1e-5)
    # Drop-last rule and the 0 / 1 region cases.
    got = bs.propagate_state_adjoint_from_last_region_input(jts, g_d, num_regions=5)
    want4 = oscan.suffix_cotangents_sequential(mats[:, :4].double(), g.double())
    assert len(got) == 5
    assert torch.allclose(torch.stack([x.cpu() for x in got], 1).double(), want4, atol=1e-5, rtol=1e-5)
    assert bs.propagate_state_adjoint_from_last_region_input([], g_d, num_regions=0) == []
    assert bs.propagate_state_adjoint_from_last_region_input(jts[:1], g_d, num_regions=1)[0] is g_d
    with pytest.raises(ValueError):
        bs.propagate_state_adjoint_from_last_region_input(jts, g_d, num_regions=4)
    one = bs.apply_jacobian_t(jts[0], g_d)
    assert torch.allclose(one.cpu(), torch.einsum("bij,bj->bi", mats[:, 0], g), atol=1e-5, rtol=1e-5)
    stats = bs.interface_state_jacobian_t_stats(jts, include_suffix=True)
    assert {"jac_local_spec_mean", "jac_suffix_spec_max"} <= set(stats)


@pytest.mark.parametrize("dtype,rank", [(torch.bfloat16, 160), (torch.float16, 192), (torch.bfloat16, 240), (torch.float16, 256)])
def test_fused_cotangents_round_as_blocked_sums(dtype, rank, device):
    """The fused cotangents of the plane kernel on random 16-bit matrices, 2-norm over the chain against fp64.  A sum of n terms of
    random sign that is rounded n times is off by about sqrt(n / 2) e of itself, e = 2.5e-8 the mean rounding of one addition.
    Summed by product steps (8 terms, then at most 16 sums) a step leaves sqrt(8 / 2 + 16 / 2) e = 0.9e-7, as one running sum of
    up to 128 terms 2.0e-7; r steps leave sqrt(r) times that, over 20 steps 2.8e-7 and 6.4e-7 on average."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents

    mats, g = oscan.make_scan_inputs(32, 20, rank, kind="randn", seed=3)
    mats = mats.to(dtype)
    _, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
    want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
    assert float((cot.cpu().double() - want).norm() / want.norm()) <= 4.2e-7


@pytest.mark.parametrize("narrow", [0, 1])
def test_forced_block_widths_in_subprocess(narrow, device):
    """LBI_SCAN_NARROW: the plane kernel on blocks of 64 columns (0) and of 32 (1), whichever the batch would get by itself, at every
    width it is built for and at one between them."""
    import os
    import subprocess
    import sys

    code = (
        "import torch, sys; sys.path.insert(0, %r);"
        "from oracle import scan as o;"
        "from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents as f;"
        "worst = 0.0\n"
        "for rank in (160, 192, 200, 256):\n"
        "    m, g = o.make_scan_inputs(3, 9, rank, kind='randn', seed=5)\n"
        "    out, cot = f(m.cuda(), g.cuda())\n"
        "    t = o.suffix_scan_sequential(m, dtype=torch.float64)\n"
        "    c = o.suffix_cotangents_sequential(m.double(), g.double())\n"
        "    worst = max(worst, float(((out.cpu().double() - t).abs().flatten(2).amax(2) / t.abs().flatten(2).amax(2)).max()))\n"
        "    worst = max(worst, float(((cot.cpu().double() - c).abs() / c.abs().amax(2, keepdim=True)).max()))\n"
        "print(worst); sys.exit(0 if 0.0 < worst <= 1e-5 else 1)"
    ) % str(Path(__file__).resolve().parents[1])
    env = dict(os.environ, LBI_SCAN_NARROW=str(narrow))
    res = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stdout + res.stderr


@pytest.mark.parametrize("kind", ["near_identity", "randn"])
def test_bf16_storage_at_the_benchmark_shape_in_both_precisions(kind, device):
    """B=64, K=128, d=256 with bf16 storage, every suffix matrix of every batch element against the sequential
    product in fp64 (on the device) and against this library's fp32 path on the same rounded inputs.  Default (suffix
    operand rounded to 16 significand bits): <= 1e-3 against fp64 and <= 2e-2 against the fp32 path, the bar for
    16-bit storage; ``exact_suffix``: the rounding of fp32 accumulation alone (<= 2e-5 over all 8192 products of 128
    factors; 1e-5 on the shorter chains of the other tests).  Both entries (column-owner kernel for the matrices alone,
    row-owner kernel with the cotangent chain), reruns bit-identical."""
    from latent_bounded_interfaces_amd.hip.interface import (suffix_scan_pullbacks,
                                                             suffix_scan_pullbacks_and_cotangents)

    bsz, count, rank = 64, 128, 256
    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind=kind, seed=11)
    mats_d, g_d = mats.to(device).to(torch.bfloat16), g.to(device)
    truth = oscan.suffix_scan_sequential(mats_d.double(), dtype=torch.float64)     # fp64 on the device
    scale = truth.abs().flatten(2).amax(dim=2).clamp_min(1e-300)

    def worst(out):
        return float(((out.double() - truth).abs().flatten(2).amax(dim=2) / scale).max())

    fp32_path = suffix_scan_pullbacks(mats_d.float())
    assert worst(fp32_path) <= 1e-5
    ref_scale = fp32_path.abs().flatten(2).amax(dim=2).clamp_min(1e-30)
    for exact, bar in ((False, 1e-3), (True, 2e-5)):
        only = suffix_scan_pullbacks(mats_d, exact_suffix=exact)
        fused, cot = suffix_scan_pullbacks_and_cotangents(mats_d, g_d, exact_suffix=exact)
        for out in (only, fused):
            err = worst(out)
            assert err <= bar, (kind, exact, err)
            assert float(((out - fp32_path).abs().flatten(2).amax(dim=2) / ref_scale).max()) <= 2e-2
            assert torch.equal(out[:, count], torch.eye(rank, device=device).expand(bsz, rank, rank))
        assert torch.equal(only, suffix_scan_pullbacks(mats_d, exact_suffix=exact)), "reruns differ"
        want = torch.einsum("bkij,bj->bki", truth, g_d.double())
        cscale = want.abs().amax(dim=2, keepdim=True).clamp_min(1e-300)
        assert float(((cot.double() - want).abs() / cscale).max()) <= 1e-5
        del only, fused, cot


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [16, 32, 48, 64, 80, 96, 128])
@pytest.mark.parametrize("bsz,count", [(1, 2), (3, 25)])
def test_cotangent_chain_off_the_grid(rank, bsz, count, dtype, device):
    """Matrices that start one element behind the allocation's grid (16-bit ones off the 4-byte words that transfers into LDS move)."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_cotangents

    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="near_identity", seed=rank + count)
    mats, g = mats.to(dtype).to(device), g.to(device)
    off = torch.empty(mats.numel() + 1, dtype=dtype, device=device)[1:].view(mats.shape).copy_(mats)
    g_off = torch.empty(g.numel() + 1, device=device)[1:].view(g.shape).copy_(g)
    assert off.data_ptr() % 16 == mats.element_size() and off.is_contiguous()
    got, again = suffix_scan_cotangents(off, g_off), suffix_scan_cotangents(mats, g)
    want = oscan.suffix_cotangents_sequential(mats.cpu().double(), g.cpu().double())
    # the bound of the test above
    bound = 2 * count * (rank + 8) * 2.0 ** -24 * float(want.norm(dim=-1).max())
    for one in (got, again):
        assert float((one.cpu().double() - want).abs().max()) <= bound


# a few small matrices each, either side of the lines between the narrow scan's chain and the scalar kernel's, alone and behind the matrices
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank,bsz,count", [(2, 4096, 2), (2, 4097, 4), (2, 4097, 5), (3, 16384, 2), (4, 16385, 1), (4, 4099, 2)])
def test_many_chains_of_a_few_small_matrices(rank, bsz, count, dtype, device):
    from latent_bounded_interfaces_amd.hip.interface import (suffix_scan_cotangents, suffix_scan_pullbacks,
                                                             suffix_scan_pullbacks_and_cotangents)

    gen = torch.Generator(device=device).manual_seed(bsz + count)
    mats = (torch.randn(bsz, count, rank, rank, generator=gen, device=device) * rank ** -0.5).to(dtype)
    g = torch.randn(bsz, rank, generator=gen, device=device)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats, g)
    assert torch.equal(out, suffix_scan_pullbacks(mats))
    eye = torch.eye(rank, device=device, dtype=torch.float64).expand(bsz, rank, rank)
    truth, want, terms = eye, g.double(), g.double().abs()
    alone = suffix_scan_cotangents(mats, g)
    for r in range(count - 1, -1, -1):
        left = mats[:, r].double()
        truth, want = left @ truth, (left @ want.unsqueeze(-1)).squeeze(-1)
        terms = (left.abs() @ terms.unsqueeze(-1)).squeeze(-1)
        # rank products and sums a step, of terms whose absolute values sum to `terms`
        bound = (count - r) * (rank + 1) * 2.0 ** -24 * terms
        assert bool(((cot[:, r].double() - want).abs() <= bound).all()) and bool(((alone[:, r].double() - want).abs() <= bound).all())
        assert float((out[:, r].double() - truth).abs().max() / truth.abs().max()) <= 1e-6
    assert torch.equal(cot[:, count], g) and torch.equal(alone[:, count], g)


# Widths up to 128 in 16 x 16 tiles: each number of row tiles with its last tile full, one short and one over, and the forms a batch
# takes: one block of 16 columns a workgroup, blocks of 32 with the vector in a workgroup of its own and beside the first block,
# chunks on either, one matrix.  Each product sums d terms in blocks of 32 (K of them one after the other): K (d / 32 + 32) roundings
# of 2^-24 against the sizes of a near-identity chain bound the error; 1e-5 is less for every case here.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank", [2, 15, 17, 31, 48, 49, 63, 64, 66, 80, 81, 96, 111, 112, 113, 128])
@pytest.mark.parametrize("bsz,count", [(1, 1), (3, 9), (2, 40), (13, 60), (44, 5), (70, 4)])
def test_narrow_scan_forms(rank, bsz, count, dtype, device):
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks, suffix_scan_pullbacks_and_cotangents

    mats, g = oscan.make_scan_inputs(bsz, count, rank, kind="near_identity", seed=rank + count)
    mats = mats.to(dtype).to(device)
    g = g.to(device)
    out, cot = suffix_scan_pullbacks_and_cotangents(mats, g)
    assert torch.equal(out, suffix_scan_pullbacks(mats))
    truth, want = torch.eye(rank, device=device, dtype=torch.float64).expand(bsz, rank, rank), g.double()
    assert torch.equal(out[:, count], torch.eye(rank, device=device).expand(bsz, rank, rank)) and torch.equal(cot[:, count], g)
    for r in range(count - 1, -1, -1):
        left = mats[:, r].double()
        truth, want = left @ truth, (left @ want.unsqueeze(-1)).squeeze(-1)
        assert float((out[:, r].double() - truth).abs().max() / truth.abs().max()) <= 1e-5
        assert float((cot[:, r].double() - want).abs().max() / want.abs().max()) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank,bsz", [(49, 90), (64, 90), (66, 70), (80, 70), (96, 70), (113, 60), (128, 60)])
def test_narrow_scan_carries_the_vector_over_several_trips(rank, bsz, dtype, device):
    """Plain chains on blocks of 32 columns with the vector beside the first block (below the twelve matrices from which on chains are cut): ten
    steps, more than two trips through the rings.  Bounds as above."""
    test_narrow_scan_forms(rank, bsz, 11, dtype, device)


# either side of the lines between the narrow scan and the 32 x 32 tiles (256 CUs), blocks of 32 columns and whole ones there
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rank,bsz", [(24, 512), (24, 513), (41, 257), (57, 128), (57, 300), (64, 300), (64, 800), (75, 40), (75, 81), (96, 81), (105, 33), (105, 65),
                                      (120, 40), (128, 65), (128, 513)])
def test_batches_at_the_lines_of_the_narrow_scan(rank, bsz, dtype, device):
    """Sums in blocks of 32 on either side: the bound above."""
    test_narrow_scan_forms(rank, bsz, 5, dtype, device)


@pytest.mark.parametrize("rank", [16, 30, 64, 77, 128])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_narrow_scan_keeps_other_rows_and_elements_apart(rank, value, device):
    """What is not finite stays where plain products put it: nothing leaks through the padding of a row's last tile."""
    from latent_bounded_interfaces_amd.hip.interface import suffix_scan_pullbacks_and_cotangents

    for bsz in (2, 70):
        mats, g = oscan.make_scan_inputs(bsz, 3, rank, kind="randn", seed=3)
        mats[0, 1, 0, rank - 1] = value
        out, cot = suffix_scan_pullbacks_and_cotangents(mats.to(device), g.to(device))
        truth = oscan.suffix_scan_sequential(mats, dtype=torch.float64)
        want = oscan.suffix_cotangents_sequential(mats.double(), g.double())
        assert torch.equal(torch.isfinite(out.cpu()), torch.isfinite(truth))
        assert torch.equal(torch.isfinite(cot.cpu()), torch.isfinite(want))
        assert torch.isfinite(out[1:]).all() and torch.isfinite(cot[1:]).all()
