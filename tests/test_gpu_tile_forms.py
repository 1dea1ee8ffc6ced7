"""The tiles that are the second form of a variant (64x64 of the 64x128 variant, 128x128 in eight waves of the 64x256
one) and the eight-wave 64x128 tile: at the edges of the tiles, with as many K blocks as stages and one more or fewer,
with every kind of K split, and grouped.

The arithmetic of an output does not depend on the tile (per K block one matrix-core dot product, folded in ascending
K, partitions summed in order), so besides the oracle's bar every result must have the bits of the 128x128 tile with
the same K split, which other tests hold to the instruction-level model.  The reference picks its tile per exact shape
(1-amd-fp8-mm/amd-fp8-mm-submission.py:528-578).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

RTOL, ATOL = 2e-2, 1e-3
FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
TILES = (4, FORM(4, 1), FORM(12, 1))


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the GPU box"
    return torch.device("cuda:0")


def _to(data, dev):
    return tuple(t.to(dev) if isinstance(t, torch.Tensor) else t for t in data)


@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (64, 64, 256), (65, 63, 384), (63, 129, 512), (128, 128, 640), (129, 127, 512), (127, 200, 768),
                                   (5, 519, 1024), (1000, 72, 384), (2051, 1030, 256), (96, 2000, 1152)])
def test_edges_and_splits(pkg, oracle, dev, m, n, k):
    cpu = pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=m, n=n, k=k)
    ref, data = oracle.ref_kernel(cpu), _to(cpu, dev)
    flag = pkg._lib.SPLIT_SUM_IN_KERNEL
    for split in (1, 2, 3, 5, 2 | flag, 3 | flag, 5 | flag):
        if split & ~flag > k // 128:
            continue
        want = pkg.custom_kernel(data, variant=3, split_k=split).clone()
        for tile in TILES:
            data[4].fill_(float("nan"))
            out = pkg.custom_kernel(data, variant=tile, split_k=split)
            what = "%dx%dx%d tile %#x split %#x" % (m, n, k, tile, split)
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), what
            ok, nbad, maxerr = oracle.within_tolerance(out, ref, RTOL, ATOL)
            assert ok, "%s: %d elements outside the bar (max abs err %g)" % (what, nbad, maxerr)


@pytest.mark.parametrize("tokens,n,k,experts,topk", [(3, 64, 128, 4, 1), (37, 200, 384, 5, 2), (150, 519, 640, 8, 3), (400, 1024, 512, 3, 2)])
def test_grouped(pkg, oracle, dev, tokens, n, k, experts, topk):
    cpu = pkg.inputs.make_grouped(pkg.inputs.CONFIGS[4], tokens=tokens, n=n, k=k, experts=experts, topk=topk)
    ref, data = oracle.ref_grouped(cpu), _to(cpu, dev)
    want = pkg.grouped_kernel(data, variant=3).clone()
    for tile in TILES:
        data[5].fill_(float("nan"))
        out = pkg.grouped_kernel(tuple(data[:5]) + (torch.full_like(data[5], float("nan")),), variant=tile)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), "tile %#x" % tile
        ok, nbad, maxerr = oracle.within_tolerance(out, ref, RTOL, ATOL)
        assert ok, "tile %#x: %d elements outside the bar (max abs err %g)" % (tile, nbad, maxerr)


def test_second_forms_are_named_and_planned(pkg, dev):
    """The plan says which form it takes, and a form that a variant does not have is refused."""
    assert (pkg.plan(512, 2048, 1024).variant, pkg.plan(512, 2048, 1024).form, pkg.plan(512, 2048, 1024).tile_n) == (4, 1, 64)
    assert (pkg.plan(4096, 1024, 4096).variant, pkg.plan(4096, 1024, 4096).form, pkg.plan(4096, 1024, 4096).tile_m) == (12, 1, 128)
    data = _to(pkg.inputs.make_dense(pkg.inputs.CONFIGS[0]), dev)
    for tile in (FORM(2, 1), FORM(4, 2), FORM(13, 0)):
        with pytest.raises(RuntimeError):
            pkg.custom_kernel(data, variant=tile, split_k=1)
