"""Grouped products of several rounds of tiles whose workgroups change places between them, with a last round that is dealt whole, cut or full."""
import pytest
import torch

from test_gpu_last_rounds import FORM, _check_grouped

pytestmark = pytest.mark.gpu


# 64x256 on 256 workgroups: 528 tiles (16 left over: cut in four), 1080 (56: in four), 700 (188: dealt whole), 420 of 70 experts, whose table is in LDS (164), 768
# (none), 540 of 270 experts, without a table (28); 64x64 on 512: four times as many, in 128 x 128 twice; 128x256 where no expert has more than 128 rows as 64x256.
@pytest.mark.parametrize("experts,n", [(33, 4096), (60, 4608), (50, 3584), (70, 1536), (64, 3072), (270, 512)])
def test_products(pkg, experts, n):
    gen = torch.Generator(device="cuda:0").manual_seed(experts)
    counts = torch.randint(1, 16, (experts,), generator=gen, device="cuda:0").tolist()
    _check_grouped(pkg, gen, counts, n, (0, 2, 12, FORM(10, 1), FORM(12, 1), FORM(4, 1)))
