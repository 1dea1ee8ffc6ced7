"""The last bytes of a and b where m or n is not a multiple of four, on every tile.

The copies' range check cuts the last one to three bytes of such an operand off, and the kernel writes them into LDS itself
(fp8bs_tiled.h).  One operand is zero but for its last four bytes, the other all ones, so that every output is a small whole
number, a lost, misplaced or doubled byte is a wrong one, and the comparison is exact.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
TILES = (2, 3, 4, FORM(4, 1), 5, 6, 9, 10, 11, 12, FORM(12, 1), FORM(12, 2), FORM(12, 3))


def _operand(rows, k, fill, shift, dev):
    """[rows, k] e4m3fn, K-major, `shift` bytes off the allocation's start; zeros but for the last four bytes, or ones."""
    raw = torch.zeros(rows * k + 16, dtype=torch.uint8, device=dev)
    flat = raw[shift:shift + rows * k]
    if fill:
        flat.fill_(0x38)                                           # 1.0
    else:
        flat[-4:] = torch.tensor([0x38, 0x40, 0x48, 0x50], dtype=torch.uint8, device=dev)      # 1, 2, 4, 8
    return flat.view(torch.float8_e4m3fn).view(k, rows).t()


@pytest.mark.parametrize("k", [128, 256, 640])
@pytest.mark.parametrize("m,n", [(1, 1), (2, 3), (3, 2), (65, 129), (129, 65), (255, 257), (257, 193), (66, 190)])
def test_last_bytes(pkg, m, n, k):
    dev = torch.device("cuda:0")
    scales = (torch.ones(k // 128, m, device=dev).t(), torch.ones(k // 128, (n + 127) // 128, device=dev).t())
    for shift in (0, 3):
        for last_of_b in (False, True):
            a, b = _operand(m, k, last_of_b, shift, dev), _operand(n, k, not last_of_b, shift, dev)
            want = (a.float() @ b.float().t()).bfloat16()
            for tile in TILES:
                if tile == 6 and (n % 8 or shift):
                    continue                                       # the streaming kernel: aligned stores and operands
                for split in (1, 2):
                    if split > k // 128:
                        continue
                    c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
                    pkg.custom_kernel((a, b, *scales, c), variant=tile, split_k=split)
                    assert torch.equal(c, want), "tile %#x split %d shift %d, last bytes of %s" % (tile, split, shift, "b" if last_of_b else "a")


@pytest.mark.parametrize("n,k", [(1, 128), (130, 256), (191, 640)])
def test_last_bytes_of_every_expert(pkg, n, k):
    """Grouped: every expert's matrix ends with bytes of its own."""
    dev = torch.device("cuda:0")
    experts, counts = 3, (5, 130, 64)
    rows = sum(counts)
    offsets = torch.tensor([0, 5, 135, 199], dtype=torch.int32, device=dev)
    a = _operand(rows, k, True, 0, dev)
    b = torch.zeros(experts, k, n, dtype=torch.uint8, device=dev)
    b.view(experts, -1)[:, -4:] = torch.tensor([[0x38, 0x40, 0x48, 0x50], [0x40, 0x38, 0x50, 0x48], [0x50, 0x48, 0x40, 0x38]], dtype=torch.uint8, device=dev)
    b = b.view(torch.float8_e4m3fn).transpose(1, 2)
    a_scale, b_scale = torch.ones(k // 128, rows, device=dev).t(), torch.ones(experts, k // 128, (n + 127) // 128, device=dev).transpose(1, 2)
    want = torch.cat([b[e].float().sum(dim=1).expand(c, n) for e, c in enumerate(counts)]).bfloat16()
    for tile in (2, 3, 4, FORM(4, 1), 9, 10, 11, 12, FORM(12, 1)):
        c = torch.full((rows, n), float("nan"), dtype=torch.bfloat16, device=dev)
        pkg.grouped_kernel((a, b, a_scale, b_scale, offsets, c), variant=tile)
        assert torch.equal(c, want), "tile %#x" % tile
