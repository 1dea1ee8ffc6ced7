"""moe.combine refuses slot_of and weights in host memory, which its kernel cannot read."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [1, 2])
def test_combine_refuses_host_tensors(which):
    moe = importlib.import_module("amd-developer-challenge-2025_amd.moe")
    args = [torch.ones(4, 128, dtype=torch.bfloat16, device="cuda:0"), torch.zeros(2, 2, dtype=torch.int32, device="cuda:0"), torch.ones(2, 2, device="cuda:0")]
    assert torch.equal(moe.combine(*args).float().cpu(), torch.full((2, 128), 2.0))
    args[which] = args[which].cpu()
    with pytest.raises(ValueError):
        moe.combine(*args)


@pytest.mark.parametrize("tokens,d", [(0, 128), (2, 0)])
def test_combine_of_nothing_takes_host_tensors(tokens, d):
    """Nothing is launched, so nothing is read."""
    moe = importlib.import_module("amd-developer-challenge-2025_amd.moe")
    out = moe.combine(torch.ones(4, d, dtype=torch.bfloat16, device="cuda:0"), torch.zeros(tokens, 2, dtype=torch.int32), torch.ones(tokens, 2))
    assert out.shape == (tokens, d) and out.is_cuda
