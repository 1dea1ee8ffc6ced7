"""Grouped products whose weights are read past the caches (fp8bs_tiled.h, MODE 6, `b_read_once`): the same bits as the 128x128 tile in eight
waves, which reads them as any other operand; nothing is written beyond c.

The operands are small whole numbers and the scales one, so every sum is exact in float32 and the comparison is of bits.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
K = 2048


def _codes(gen, *shape):
    values = torch.tensor([0x00, 0x38, 0xB8, 0x40], dtype=torch.uint8, device="cuda:0")          # 0, 1, -1, 2
    return values[torch.randint(4, shape, generator=gen, device="cuda:0", dtype=torch.int32)].view(torch.float8_e4m3fn)


def _case(experts, n, counts):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(experts + n)
    rows = sum(counts)
    a, b = _codes(gen, K, rows).t(), _codes(gen, experts, K, n).transpose(1, 2)
    b_scale = torch.ones(experts, K // 128, (n + 127) // 128, device=dev).transpose(1, 2)
    offsets = torch.tensor([0, *counts], device=dev).cumsum(0).int()
    return a, b, torch.ones(K // 128, rows, device=dev).t(), b_scale, offsets


# Weights just over the 256 MiB line, rows of b whole lines and not (which are read as before): one row an expert (an odd number of rows of a: the
# instantiation with tails), 48 (the line of the tile of 64 rows), 192 (the line of the tile of 256), and an expert that holds most of the
# rows, whose weights are read more than once.
@pytest.mark.parametrize("n", [4096, 4104])
@pytest.mark.parametrize("counts", [[1] * 33, [48] * 33, [192] * 33, [0, 701] + [7] * 31])
def test_grouped(pkg, n, counts):
    a, b, a_scale, b_scale, offsets = _case(33, n, counts)
    assert b.numel() >= 256 << 20
    rows = sum(counts)
    want = torch.full((rows + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    pkg.grouped_kernel((a, b, a_scale, b_scale, offsets, want[:rows]), variant=FORM(12, 1))
    bounds, e = offsets.tolist(), 5
    assert torch.equal(want[bounds[e]:bounds[e + 1]], (a[bounds[e]:bounds[e + 1]].float() @ b[e].float().t().contiguous()).bfloat16())
    for variant in (0, 2, 12):
        c = torch.full((rows + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
        pkg.grouped_kernel((a, b, a_scale, b_scale, offsets, c[:rows]), variant=variant)
        assert torch.equal(c.view(torch.int16), want.view(torch.int16)), "variant %d" % variant


@pytest.mark.parametrize("n", [4096, 4224])
def test_grouped_silu_mul(pkg, n):
    counts = [3, 0, 31] + [15] * 30
    a, b, a_scale, b_scale, offsets = _case(33, n, counts)
    rows, lib, out = sum(counts), pkg._lib.load(), []
    for variant in (4, 2, 12):
        h = torch.full((rows, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda:0")
        pkg._lib.check(lib.fp8bs_gemm_silu_mul_ws(a.data_ptr(), b.data_ptr(), a_scale.data_ptr(), b_scale.data_ptr(), h.data_ptr(), offsets.data_ptr(), 33, rows, n, K, variant, 1,
                                                  None, 0, torch.cuda.current_stream().cuda_stream))
        out.append(h.view(torch.int16))
        assert not torch.isnan(h).any()
    assert torch.equal(out[1], out[0]) and torch.equal(out[2], out[0])
