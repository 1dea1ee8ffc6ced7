"""Rounds of tiles that do not fill the chip: dealt to all XCDs, and tiles of 256 columns cut in two or four by columns where they
leave half of it, or three quarters, idle (fp8bs_tiled.h, `place` and `take_part`); and the grouped walk with its table in
registers (up to 64 experts), in LDS, and past that.

The operands are small whole numbers and the scales powers of two that differ from block to block of columns, so every output is
exact in float32 and the comparison is of bits; c starts as NaN, so that a part left out shows.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
K = 256


def _codes(gen, *shape):
    values = torch.tensor([0x00, 0x38, 0xB8, 0x40], dtype=torch.uint8, device="cuda:0")          # 0, 1, -1, 2
    return values[torch.randint(4, shape, generator=gen, device="cuda:0")].view(torch.float8_e4m3fn)


def _column_scales(n, dev):
    """[K/128, ceil(n/128)]: 1, 2 and 4 in turn over the blocks of columns, and their expansion to [n]."""
    s = torch.exp2((torch.arange((n + 127) // 128, device=dev) % 3).float())
    return s.expand(K // 128, -1).contiguous(), s.repeat_interleave(128)[:n]


# Tiles beyond the last full round of 256 or 512 workgroups: 256x256: 324 tiles (68 left over), 320 (64), the last tile 250 or 10 columns
# wide; 64x256: 576 (64 left over, the last tile 10 columns wide) and 648 (136).  The last two: 3100 tiles, 28 of them behind twelve full
# rounds, where the last round is neither spread nor cut.
@pytest.mark.parametrize("tile,m,n", [(2, 4608, 4608), (2, 5111, 4090), (2, 5120, 3850), (12, 2304, 3850), (12, 2300, 4601), (2, 12790, 15810), (12, 3190, 15810)])
def test_dense(pkg, tile, m, n):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m + n)
    a, b = _codes(gen, K, m).t(), _codes(gen, K, n).t()
    b_scale, columns = _column_scales(n, dev)
    c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    pkg.custom_kernel((a, b, torch.ones(K // 128, m, device=dev).t(), b_scale.t(), c), variant=tile)
    assert torch.equal(c, (a.float() @ b.float().t().contiguous() * columns).bfloat16())


def _check_grouped(pkg, gen, counts, n, tiles):
    dev = torch.device("cuda:0")
    rows, experts = sum(counts), len(counts)
    offsets = torch.tensor([0, *counts], device=dev).cumsum(0).int()
    a, b = _codes(gen, K, rows).t(), _codes(gen, experts, K, n).transpose(1, 2)
    b_scale, columns = _column_scales(n, dev)
    b_scale = b_scale.expand(experts, -1, -1).contiguous().transpose(1, 2)
    bounds = offsets.tolist()
    want = torch.cat([a[lo:hi].float() @ b[e].float().t().contiguous() * columns for e, (lo, hi) in enumerate(zip(bounds, bounds[1:]))]).bfloat16()
    for tile in tiles:
        c = torch.full((rows, n), float("nan"), dtype=torch.bfloat16, device=dev)
        pkg.grouped_kernel((a, b, torch.ones(K // 128, rows, device=dev).t(), b_scale, offsets, c), variant=tile)
        assert torch.equal(c, want), "tile %#x" % tile


@pytest.mark.parametrize("experts", [1, 3, 63, 64, 65, 300])
@pytest.mark.parametrize("n", [70, 250, 266, 520])
def test_grouped(pkg, experts, n):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(experts * 1000 + n)
    counts = torch.randint(0, 40, (experts,), generator=gen, device=dev).mul_(torch.rand(experts, generator=gen, device=dev) < 0.7).tolist()
    counts[-1] += 131                                              # several tiles of one expert
    _check_grouped(pkg, gen, counts, n, (0, 2, 3, 12, FORM(12, 1)))


# Few rows an expert, several rounds of 256 or 512 tiles: the workgroups of an XCD change places between them.  64x256: 528 tiles (16 left over), 768 (none),
# 1080 (56), 700 (188 left over, not cut), 490 of 70 experts, whose table is in LDS (234, not cut); 64x64: 1890 to 4320.
@pytest.mark.parametrize("experts,n", [(33, 4090), (48, 4096), (60, 4601), (50, 3500), (70, 1700)])
def test_grouped_across_the_experts_in_rounds(pkg, experts, n):
    gen = torch.Generator(device="cuda:0").manual_seed(experts)
    counts = torch.randint(1, 16, (experts,), generator=gen, device="cuda:0").tolist()
    _check_grouped(pkg, gen, counts, n, (0, 2, 12, FORM(12, 1), FORM(4, 1)))


@pytest.mark.parametrize("tile,counts", [(2, (4100, 0, 5000, 3700)), (12, (1030, 0, 1250, 920))])
def test_grouped_of_many_rounds(pkg, tile, counts):
    """Some 3300 tiles: the last round behind twelve full ones."""
    _check_grouped(pkg, torch.Generator(device="cuda:0").manual_seed(tile), counts, 15810, (tile,))


def _silu_mul(pkg, a, b, a_scale, b_scale, offsets, rows, n, variant):
    """gate_up_silu with the tile forced, unsplit; h starts as NaN."""
    lib = pkg._lib.load()
    h = torch.full((rows, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    pkg._lib.check(lib.fp8bs_gemm_silu_mul_ws(a.data_ptr(), b.data_ptr(), a_scale.data_ptr(), b_scale.data_ptr(), h.data_ptr(), None if offsets is None else offsets.data_ptr(),
                                              0 if offsets is None else offsets.numel() - 1, rows, n, K, variant, 1, None, 0, torch.cuda.current_stream().cuda_stream))
    assert not torch.isnan(h).any()
    return h.view(torch.int16)


# n/2 on the 8-column grid and off it, the last tile 10 columns wide in two of them.  64x128 is never cut.
@pytest.mark.parametrize("tile,m,n", [(2, 4608, 4608), (2, 5111, 4090), (2, 5120, 3850), (12, 2304, 3850), (12, 2300, 4602)])
def test_dense_silu_mul(pkg, tile, m, n):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m + n)
    a, b = _codes(gen, K, m).t(), _codes(gen, K, n).t()
    data = (a, b, torch.ones(K // 128, m, device=dev).t(), _column_scales(n, dev)[0].t(), None, m, n)
    assert torch.equal(_silu_mul(pkg, *data, tile), _silu_mul(pkg, *data, 4))


@pytest.mark.parametrize("experts", [1, 3, 64, 65])
@pytest.mark.parametrize("n", [70, 250, 266, 520])
def test_grouped_silu_mul(pkg, experts, n):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(experts * 1000 + n)
    counts = torch.randint(0, 40, (experts,), generator=gen, device=dev).tolist()
    counts[-1] += 131
    rows = sum(counts)
    a, b = _codes(gen, K, rows).t(), _codes(gen, experts, K, n).transpose(1, 2)
    b_scale = _column_scales(n, dev)[0].expand(experts, -1, -1).contiguous().transpose(1, 2)
    data = (a, b, torch.ones(K // 128, rows, device=dev).t(), b_scale, torch.tensor([0, *counts], device=dev).cumsum(0).int(), rows, n)
    want = _silu_mul(pkg, *data, 4)
    for tile in (2, 12):
        assert torch.equal(_silu_mul(pkg, *data, tile), want), "tile %d" % tile
