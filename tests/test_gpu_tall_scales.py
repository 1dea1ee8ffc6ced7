"""Grouped calls on the 128x256 tile with scales that differ by row, K block, block of columns and expert: its stage holds two waves' rows of a_scale and the b_scale
of two blocks of columns, and a wave takes one of these.  At the edges of the tile, with fewer K blocks than stages and more, aligned and not, and with the
experts found in registers, in the table in LDS and past that.

The operands are small whole numbers and the scales powers of two: every sum is a multiple of 1/4 below 2^15, exact in float32 in any order, and the comparison is of bits.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

TALL, OTHER = 10 | 2 << 8, 12 | 2 << 8                           # FP8BS_VARIANT_FORM(10, 1) and (12, 1)


def _codes(gen, *shape):
    values = torch.tensor([0x00, 0x38, 0xB8, 0x40], dtype=torch.uint8, device="cuda:0")          # 0, 1, -1, 2
    return values[torch.randint(4, shape, generator=gen, device="cuda:0", dtype=torch.int32)].view(torch.float8_e4m3fn)


def _case(n, k, counts):
    dev, experts, rows = torch.device("cuda:0"), len(counts), sum(counts)
    gen = torch.Generator(device=dev).manual_seed(experts + n + k)
    scales = lambda *shape: torch.exp2(torch.randint(-1, 2, shape, generator=gen, device=dev).float())      # 1/2, 1, 2
    a, b = _codes(gen, k, rows).t(), _codes(gen, experts, k, n).transpose(1, 2)
    return a, b, scales(k // 128, rows).t(), scales(experts, k // 128, (n + 127) // 128).transpose(1, 2), torch.tensor([0, *counts], device=dev).cumsum(0).int()


def _counts(experts):
    gen = torch.Generator().manual_seed(experts)
    return (torch.randint(0, 30, (experts,), generator=gen) * (torch.rand(experts, generator=gen) < 0.8)).tolist() + [131]


EDGES = [(512, 1024, (0, 1, 63, 64, 65, 127)), (256, 128, (128, 129, 4)), (776, 256, (257, 0, 31, 300)), (1027, 384, (130, 66, 5)), (130, 1152, (70, 200)), (1, 256, (3, 140))]


@pytest.mark.parametrize("n,k,counts", EDGES + [(520, 256, _counts(e)) for e in (63, 64, 70, 127, 262, 263, 400)])
def test_grouped(pkg, n, k, counts):
    a, b, a_scale, b_scale, offsets = _case(n, k, counts)
    rows, bounds = sum(counts), offsets.tolist()
    want = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda:0")
    scaled = a.float() * a_scale.repeat_interleave(128, 1)
    for e, (lo, hi) in enumerate(zip(bounds, bounds[1:])):
        weights = b[e].float() * b_scale[e].repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
        want[lo:hi] = (scaled[lo:hi] @ weights.t().contiguous()).bfloat16()
    c = torch.full((rows + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    pkg.grouped_kernel((a, b, a_scale, b_scale, offsets, c[:rows]), variant=TALL)
    assert torch.equal(c[:rows], want) and torch.isnan(c[rows]).all()


@pytest.mark.parametrize("n,k,counts", [case for case in EDGES if case[0] % 2 == 0] + [(4096, 2048, (20, 70, 0, 129) + (33,) * 34)])
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
