"""Grouped calls on the 128x256 tile (FP8BS_VARIANT_FORM(10, 1)): the same bits as the 128x128 tile in eight waves, nothing written beyond c,
with weights that are read past the caches and with smaller ones; aligned and not.

The operands are small whole numbers and the scales one, so every sum is exact in float32 and the comparison is of bits.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
TALL, OTHER = FORM(10, 1), FORM(12, 1)


def _codes(gen, *shape):
    values = torch.tensor([0x00, 0x38, 0xB8, 0x40], dtype=torch.uint8, device="cuda:0")          # 0, 1, -1, 2
    return values[torch.randint(4, shape, generator=gen, device="cuda:0", dtype=torch.int32)].view(torch.float8_e4m3fn)


def _case(n, k, counts):
    dev, experts, rows = torch.device("cuda:0"), len(counts), sum(counts)
    gen = torch.Generator(device=dev).manual_seed(experts + n)
    a, b = _codes(gen, k, rows).t(), _codes(gen, experts, k, n).transpose(1, 2)
    b_scale = torch.ones(experts, k // 128, (n + 127) // 128, device=dev).transpose(1, 2)
    offsets = torch.tensor([0, *counts], device=dev).cumsum(0).int()
    return a, b, torch.ones(k // 128, rows, device=dev).t(), b_scale, offsets


# No row, one, the edges of a wave's rows and of a tile's; experts that start on any row; the last column tile whole, of a few columns and odd
# (the instantiation with tails); one K block, fewer than the stages, more; and 33 experts whose weights pass the 256 MiB line.
@pytest.mark.parametrize("n,k,counts", [(512, 1024, (0, 1, 63, 64, 65, 127)), (256, 128, (128, 129, 4)), (776, 256, (257, 0, 31, 300)), (1027, 384, (130, 66, 5)),
                                        (4096, 2048, (20, 70, 0, 129) + (33,) * 29), (4224, 2048, (61,) * 33)])
def test_grouped(pkg, n, k, counts):
    a, b, a_scale, b_scale, offsets = _case(n, k, counts)
    rows, out = sum(counts), []
    for variant in (OTHER, TALL):
        c = torch.full((rows + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
        pkg.grouped_kernel((a, b, a_scale, b_scale, offsets, c[:rows]), variant=variant)
        out.append(c.view(torch.int16))
        assert torch.isnan(c[rows]).all() and not torch.isnan(c[:rows]).any()
    assert torch.equal(out[0], out[1])
    bounds, e = offsets.tolist(), max(range(len(counts)), key=counts.__getitem__)
    want = (a[bounds[e]:bounds[e + 1]].float() @ b[e].float().t().contiguous()).bfloat16()
    assert torch.equal(out[1][bounds[e]:bounds[e + 1]], want.view(torch.int16))


@pytest.mark.parametrize("n,k,counts", [(512, 512, (0, 1, 65, 129)), (388, 256, (70, 33)), (4096, 2048, (20, 70, 0, 129) + (33,) * 29)])
def test_grouped_silu_mul(pkg, n, k, counts):
    a, b, a_scale, b_scale, offsets = _case(n, k, counts)
    rows, lib, out = sum(counts), pkg._lib.load(), []
    for variant in (OTHER, TALL):
        h = torch.full((rows, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda:0")
        pkg._lib.check(lib.fp8bs_gemm_silu_mul_ws(a.data_ptr(), b.data_ptr(), a_scale.data_ptr(), b_scale.data_ptr(), h.data_ptr(), offsets.data_ptr(), len(counts), rows, n, k, variant, 1,
                                                  None, 0, torch.cuda.current_stream().cuda_stream))
        out.append(h.view(torch.int16))
        assert not torch.isnan(h).any()
    assert torch.equal(out[0], out[1])
