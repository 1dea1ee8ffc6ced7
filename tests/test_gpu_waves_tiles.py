"""The small tiles whose eight waves each hold a K partition (forms 2 and 3 of the 64x256 variant: 16x64 and 32x64): at the edges
of the tiles, with fewer K blocks than waves (unsplit: folded in order where the waves meet), uneven and empty partitions, odd sizes and operands
on any byte.

The arithmetic is the K split's - one matrix-core dot product per K block, folded in ascending K, partitions added in order - so
every result must have the bits of the 128x128 tile with the same split and the reduce kernel.  The reference picks its
tile per exact shape (1-amd-fp8-mm/amd-fp8-mm-submission.py:528-578).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
TILES = (FORM(12, 2), FORM(12, 3))


def _bits(t):
    return t.view(torch.int16)


def _operands(pkg, m, n, k):
    return tuple(t.to("cuda:0") for t in pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=m, n=n, k=k))


@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (16, 64, 384), (17, 65, 512), (31, 63, 1024), (33, 129, 1152), (5, 519, 1664), (100, 1001, 2048),
                                   (257, 130, 640), (64, 2050, 896), (1023, 70, 1280), (15, 3, 3072)])
def test_edges_and_splits(pkg, oracle, m, n, k):
    data = _operands(pkg, m, n, k)
    ref = oracle.ref_kernel(tuple(t.cpu() for t in data))
    for split in (1, 2, 3, 5, 7, 8):
        if split > k // 128:
            continue
        want = pkg.custom_kernel(data, variant=3, split_k=split).clone()
        for tile in TILES:
            data[4].fill_(float("nan"))
            out = pkg.custom_kernel(data, variant=tile, split_k=split)
            assert torch.equal(_bits(out), _bits(want)), "tile %#x split %d" % (tile, split)
            ok, nbad, maxerr = oracle.within_tolerance(out, ref, 2e-2, 1e-3)
            assert ok, "tile %#x split %d: %d elements outside the bar (max abs err %g)" % (tile, split, nbad, maxerr)


@pytest.mark.parametrize("m,n,k,shift", [(37, 190, 1024, 1), (61, 257, 640, 3), (20, 128, 1280, 2)])
def test_operands_on_any_byte_and_a_guarded_output(pkg, m, n, k, shift):
    a, b, sa, sb, _ = _operands(pkg, m, n, k)
    raw = lambda t, nbytes: torch.cat([torch.zeros(shift, dtype=torch.uint8, device=t.device), t.t().contiguous().view(torch.uint8).flatten()])[shift:].view(torch.uint8)
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    ra, rb = raw(a, m * k), raw(b, n * k)
    want = pkg.custom_kernel((a, b, sa, sb, torch.empty(m, n, dtype=torch.bfloat16, device=a.device)), variant=3, split_k=4)
    for tile in TILES:
        out = torch.full((m * n + 64,), 7.0, dtype=torch.bfloat16, device=a.device)
        st = lib.fp8bs_gemm_ex(ra.data_ptr(), rb.data_ptr(), sa.data_ptr(), sb.data_ptr(), out.data_ptr() + 2 * 33, None, 0, m, n, k, tile, 4, stream)
        assert st == 0
        assert torch.equal(_bits(out[33:33 + m * n].view(m, n)), _bits(want))
        assert bool((out[:33] == 7).all()) and bool((out[33 + m * n:] == 7).all())           # nothing written outside c


@pytest.mark.parametrize("m,n,k", [(1, 2, 384), (33, 130, 640), (250, 512, 1024), (64, 1030, 2048)])
def test_silu_mul(pkg, m, n, k):
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    a, b, sa, sb, _ = _operands(pkg, m, n, k)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=a.device)

    def run(tile, split, ws_bytes):
        h = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device=a.device)
        assert lib.fp8bs_gemm_silu_mul_ws(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), h.data_ptr(), None, 0, m, n, k, tile, split,
                                          ws.data_ptr() if ws_bytes else None, ws_bytes, stream) == 0
        return h
    for split in (1, 3, 8):
        if split <= k // 128:
            want = run(2, split, ws.numel())
            for tile in TILES:
                assert torch.equal(_bits(run(tile, split, 0)), _bits(want)), "tile %#x split %d" % (tile, split)


def test_planned_forced_and_refused(pkg):
    lib = pkg._lib.load()
    for m, n, k in [(256, 512, 1024), (49, 1280, 1024), (1, 1088, 1664), (64, 512, 2048)]:
        p = pkg.plan(m, n, k)
        assert (p.variant, p.tile_n) == (12, 64) and p.form in (2, 3) and p.split_k == (1 if k <= 1024 else 8)
        data = _operands(pkg, m, n, k)
        want = pkg.custom_kernel(data, variant=3, split_k=p.split_k).clone()
        data[4].fill_(float("nan"))
        assert torch.equal(_bits(pkg.custom_kernel(data)), _bits(want))
        for split in (2, 16 if k >= 2048 else 4):                 # the tile left to the library, the split forced: any number
            assert torch.equal(_bits(pkg.custom_kernel(data, split_k=split)), _bits(pkg.custom_kernel(data, variant=3, split_k=split).clone()))
        a, b, sa, sb, c = data
        args = (a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr())
        assert lib.fp8bs_gemm(*args, None, 0, m, n, k, None) == 0                                  # no workspace
        assert lib.fp8bs_gemm_ex(*args, None, 0, m, n, k, TILES[0], -1, None) == 7
        if k // 128 > 8:
            assert lib.fp8bs_gemm_ex(*args, None, 0, m, n, k, TILES[0], 9, None) == 7
        ro = torch.tensor([0, m], dtype=torch.int32, device=a.device)
        assert lib.fp8bs_gemm_grouped_ex(*args, ro.data_ptr(), 1, m, n, k, TILES[0], None) == 7
    torch.cuda.synchronize()
