"""Grouped products of more than 288 MiB of weights (fp8bs_tiled.h, MODE 6): experts of one row of tiles, whose weights are read past the caches, beside experts
of several and of none; with the experts' table in registers, in LDS and past that; scales that differ by row, K block, block of columns and expert.

The operands are small whole numbers and the scales powers of two: every sum is a multiple of 1/4 below 2^16, exact in float32 in any order, and the comparison is of bits.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
TILES = (0, 2, 12, FORM(10, 1))


def _codes(gen, *shape):
    values = torch.tensor([0x00, 0x38, 0xB8, 0x40], dtype=torch.uint8, device="cuda:0")          # 0, 1, -1, 2
    return values[torch.randint(4, shape, generator=gen, device="cuda:0", dtype=torch.int32)].view(torch.float8_e4m3fn)


def _scales(gen, *shape):
    return torch.exp2(torch.randint(-1, 2, shape, generator=gen, device="cuda:0").float())       # 1/2, 1, 2


# 37 experts of 8 MiB: one row each (an odd number of rows of a), a hot one beside few rows, two rows of tiles of each height, none of some so
# that what is read is 280 MiB and less; 100 of 3 MiB and 270 of 1.125 MiB.
@pytest.mark.parametrize("n,k,counts", [(4096, 2048, [1] * 37), (4096, 2048, [5, 900, 0] + [9] * 35), (4096, 2048, [65, 129, 257, 64, 128, 256] + [30] * 31),
                                        (4096, 2048, [8, 0] + [40] * 34 + [0, 0]), (2048, 1536, [20, 300, 0] + [11] * 97), (1024, 1152, [70, 0, 1, 400] + [7] * 266)])
def test_products(pkg, n, k, counts):
    dev, experts, rows = torch.device("cuda:0"), len(counts), sum(counts)
    gen = torch.Generator(device=dev).manual_seed(rows + n)
    a, b = _codes(gen, k, rows).t(), _codes(gen, experts, k, n).transpose(1, 2)
    a_scale, b_scale = _scales(gen, k // 128, rows).t(), _scales(gen, experts, k // 128, n // 128).transpose(1, 2)
    offsets = torch.tensor([0, *counts], device=dev).cumsum(0).int()
    assert b.numel() >= 288 << 20
    want, bounds = torch.empty(rows, n, dtype=torch.bfloat16, device=dev), offsets.tolist()
    scaled = a.float() * a_scale.repeat_interleave(128, 1)
    for e, (lo, hi) in enumerate(zip(bounds, bounds[1:])):
        weights = b[e].float() * b_scale[e].repeat_interleave(128, 0).repeat_interleave(128, 1)
        want[lo:hi] = (scaled[lo:hi] @ weights.t().contiguous()).bfloat16()
    for variant in TILES:
        c = torch.full((rows + 1, n), float("nan"), dtype=torch.bfloat16, device=dev)
        pkg.grouped_kernel((a, b, a_scale, b_scale, offsets, c[:rows]), variant=variant)
        assert torch.equal(c[:rows], want), "variant %#x" % variant
        assert torch.isnan(c[rows]).all()
