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


def _grouped_ws(lib, data, variant, split, ws, silu_out=None):
    a, b, sa, sb, ro, c = data
    out = c if silu_out is None else silu_out
    fn = lib.fp8bs_gemm_grouped_ws if silu_out is None else lib.fp8bs_gemm_silu_mul_ws
    st = fn(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), out.data_ptr(), ro.data_ptr(), b.shape[0], a.shape[0], b.shape[1], b.shape[2],
            variant, split, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.fp8bs_strerror(st)
    return out


@pytest.mark.parametrize("tokens,n,k,experts,topk", [(1, 64, 256, 8, 2), (37, 200, 384, 5, 2), (150, 518, 640, 8, 3), (90, 300, 1152, 4, 4)])
def test_grouped_k_split(pkg, oracle, dev, tokens, n, k, experts, topk):
    """The grouped walk in K partitions, plain and with the silu-mul epilogue: every tile that has the form gives the same
    bits (whatever the workspace holds), plain ones within the oracle's bar; replays of a captured launch start clean."""
    lib = pkg._lib.load()
    cpu = pkg.inputs.make_grouped(pkg.inputs.CONFIGS[4], tokens=tokens, n=n, k=k, experts=experts, topk=topk)
    ref, data = oracle.ref_grouped(cpu), _to(cpu, dev)
    ws = torch.randint(0, 256, (64 << 20,), dtype=torch.uint8, device=dev)
    rows = data[0].shape[0]
    for split in (2, 3, 7):
        if split > k // 128:
            continue
        want = want_h = None
        for tile in (12, FORM(12, 1), FORM(4, 1)):
            what = "tile %#x split %d" % (tile, split)
            out = _grouped_ws(lib, data[:5] + (torch.full_like(data[5], float("nan")),), tile, split, ws)
            h = _grouped_ws(lib, data, tile, split, ws, torch.full((rows, n // 2), float("nan"), dtype=torch.bfloat16, device=dev))
            ok, nbad, maxerr = oracle.within_tolerance(out, ref, RTOL, ATOL)
            assert ok, "%s: %d elements outside the bar (max abs err %g)" % (what, nbad, maxerr)
            # (the epilogue works on the unrounded sums: its own rounding, and the two bf16 roundings in this reference)
            g = out.float()
            href = torch.nn.functional.silu(g[:, 0::2]) * g[:, 1::2]
            assert bool(((h.float() - href).abs() <= ATOL + 2 * RTOL * href.abs()).all()), what
            assert want is None or torch.equal(out.view(torch.int16), want.view(torch.int16)), what
            assert want_h is None or torch.equal(h.view(torch.int16), want_h.view(torch.int16)), what
            want, want_h = out, h
    graph = torch.cuda.CUDAGraph()
    out = torch.empty_like(data[5])
    _grouped_ws(lib, data[:5] + (out,), 12, 2, ws)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        _grouped_ws(lib, data[:5] + (out,), 12, 2, ws)
    first = _grouped_ws(lib, data[:5] + (torch.empty_like(out),), 12, 2, ws)
    for _ in range(3):
        out.fill_(5.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), first.view(torch.int16))
        pkg.grouped_kernel(data)
        torch.cuda.synchronize()
    need = ws.numel()
    for tile, split in ((2, 2), (3, 2)):                              # tiles without the form
        a, b, sa, sb, ro, c = data
        assert lib.fp8bs_gemm_grouped_ws(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr(), ro.data_ptr(), experts, rows, n, k,
                                         tile, split, ws.data_ptr(), need, None) == 7


@pytest.mark.parametrize("m,n,k", [(1, 2, 128), (65, 130, 384), (250, 512, 1024), (127, 262, 640), (64, 1030, 896), (300, 96, 512)])
def test_dense_silu_mul_on_every_tile_and_split(pkg, dev, m, n, k):
    """The epilogue on every tile that has it, unsplit, summed in the kernel and in the reduce kernel: the bits of the
    256x256 tile's with the same K split."""
    lib = pkg._lib.load()
    flag = pkg._lib.SPLIT_SUM_IN_KERNEL
    a, b, sa, sb, _ = _to(pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=m, n=n, k=k), dev)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)

    def run(tile, split):
        h = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device=dev)
        st = lib.fp8bs_gemm_silu_mul_ws(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), h.data_ptr(), None, 0, m, n, k, tile, split,
                                        ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
        assert st == 0, lib.fp8bs_strerror(st)
        return h
    for split in (1, 2, 3, 5):
        if split > k // 128:
            continue
        want = run(2, split)
        for tile in (10, 4, FORM(4, 1), 12, FORM(12, 1)):
            for form in (0, flag) if split > 1 else (0,):
                assert torch.equal(run(tile, split | form).view(torch.int16), want.view(torch.int16)), "tile %#x split %#x" % (tile, split | form)
    assert lib.fp8bs_gemm_silu_mul_ws(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), a.data_ptr(), None, 0, m, n, k, 11, 1,
                                      ws.data_ptr(), ws.numel(), None) == 7          # a tile without the epilogue


def test_second_forms_are_named_and_planned(pkg, dev):
    """The plan says which form it takes, and a form that a variant does not have is refused."""
    assert (pkg.plan(512, 2048, 1024).variant, pkg.plan(512, 2048, 1024).form, pkg.plan(512, 2048, 1024).tile_n) == (4, 1, 64)
    assert (pkg.plan(4096, 1024, 4096).variant, pkg.plan(4096, 1024, 4096).form, pkg.plan(4096, 1024, 4096).tile_m) == (12, 1, 128)
    data = _to(pkg.inputs.make_dense(pkg.inputs.CONFIGS[0]), dev)
    for tile in (FORM(2, 1), FORM(4, 2), FORM(13, 0)):
        with pytest.raises(RuntimeError):
            pkg.custom_kernel(data, variant=tile, split_k=1)


def test_grouped_split_keeps_to_its_workspace_with_a_malformed_table(pkg, dev):
    """Row offsets that descend claim more tiles than the rows can give: the partial tiles stay inside the workspace."""
    lib = pkg._lib.load()
    experts, n, k = 6, 256, 512
    data = _to(pkg.inputs.make_grouped(pkg.inputs.CONFIGS[4], tokens=96, n=n, k=k, experts=experts, topk=2), dev)
    rows = data[0].shape[0]
    table = torch.tensor([0, rows, 0, rows, 0, rows, 0], dtype=torch.int32, device=dev)
    for tile, bm, bn in ((12, 64, 256), (FORM(12, 1), 128, 128), (FORM(4, 1), 64, 64)):
        need = 16384 + (experts + rows // (bm - 14)) * (n // bn) * 2 * bm * bn * 4        # a header and two partial tiles per tile
        ws = torch.full((need + (8 << 20),), 0xA5, dtype=torch.uint8, device=dev)
        _grouped_ws(lib, data[:4] + (table, torch.empty_like(data[5])), tile, 2, ws[:need])
        assert bool((ws[need:] == 0xA5).all()), "tile %#x" % tile


def test_captured_calls_keep_no_buffer_of_the_table(pkg, dev):
    """A captured K split works in memory of its graph: a larger call, which outgrows the tables' buffers, and the caching
    allocator's reuse of them leave the replays as they were."""
    sub = __import__("importlib").import_module(pkg.__name__ + ".submission")
    moe = __import__("importlib").import_module(pkg.__name__ + ".moe")
    grouped = _to(pkg.inputs.make_grouped(pkg.inputs.CONFIGS[4], tokens=8, n=512, k=7168, experts=8, topk=2), dev)
    dense = _to(pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=64, n=512, k=7168), dev)
    idx = torch.stack([torch.randperm(16)[:4] for _ in range(2048)]).to(torch.int32).to(dev)
    assert pkg.plan(64, 512, 7168).workspace_bytes > 0
    assert pkg._lib.load().fp8bs_grouped_workspace_bytes(8, grouped[0].shape[0], 512, 7168) > 0

    def calls():
        pkg.custom_kernel(dense)
        pkg.grouped_kernel(grouped)
        return (dense[4], grouped[5]) + tuple(moe.route(idx, 16))
    want = [t.clone() for t in calls()]
    torch.cuda.synchronize()
    before = {k: v.data_ptr() for k, v in sub._workspaces.items()}, {k: v.data_ptr() for k, v in moe._route_ws.items()}
    held = sum(map(len, sub._held.values()))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = calls()
    assert held == sum(map(len, sub._held.values()))
    assert before == ({k: v.data_ptr() for k, v in sub._workspaces.items()}, {k: v.data_ptr() for k, v in moe._route_ws.items()})
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for t, w in zip(out, want):
            assert torch.equal(t.view(torch.int16), w.view(torch.int16))
        sub._workspaces.clear()
        moe._route_ws.clear()
        pkg.custom_kernel(dense, split_k=7)
        torch.full((32 << 20,), 255, dtype=torch.uint8, device=dev)
        torch.cuda.synchronize()


def test_a_capture_begun_with_hip_itself(pkg, dev):
    """No memory pool belongs to such a graph: its replays stay right when larger calls outgrow the stream's buffers and the
    allocator hands out what was freed, with eager work between them."""
    import ctypes
    moe = __import__("importlib").import_module(pkg.__name__ + ".moe")
    hip = ctypes.CDLL("libamdhip64.so")
    def ok(status):
        assert status == 0, "HIP status %d" % status
    dense = _to(pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=64, n=512, k=7168), dev)
    idx = torch.stack([torch.randperm(16)[:4] for _ in range(2048)]).to(torch.int32).to(dev)
    out = (torch.empty(17, dtype=torch.int32, device=dev), torch.empty(8192, dtype=torch.int32, device=dev), torch.empty(2048, 4, dtype=torch.int32, device=dev))
    assert pkg.plan(64, 512, 7168).workspace_bytes > 0

    def calls():
        pkg.custom_kernel(dense)
        moe.route(idx, 16, out=out)
    side = torch.cuda.Stream()
    graph, program = ctypes.c_void_p(), ctypes.c_void_p()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        calls()
        torch.cuda.synchronize()
        want = [t.clone() for t in (dense[4],) + out]
        torch.cuda.synchronize()
        stream = ctypes.c_void_p(side.cuda_stream)
        ok(hip.hipStreamBeginCapture(stream, 2))                     # relaxed
        try:
            calls()
        finally:
            ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)))
        ok(hip.hipGraphInstantiate(ctypes.byref(program), graph, None, None, 0))
        for _ in range(3):
            for t in (dense[4],) + out:
                t.zero_()
            ok(hip.hipGraphLaunch(program, stream))
            torch.cuda.synchronize()
            for t, w in zip((dense[4],) + out, want):
                assert torch.equal(t, w)
            pkg.custom_kernel(dense, split_k=56)
            moe.route(idx.repeat(64, 1), 16)
            kept = [torch.full((size,), 255, dtype=torch.uint8, device=dev) for size in (1 << 20, 2 << 20, 4 << 20, 8 << 20)]
            ok(hip.hipGraphLaunch(program, stream))
            torch.cuda.synchronize()
            assert all(bool((t == 255).all()) for t in kept)         # nothing was written to memory that is another's now
        ok(hip.hipGraphExecDestroy(program))
        ok(hip.hipGraphDestroy(graph))


def test_grouped_split_with_the_tile_left_to_the_library(pkg, dev):
    """A split given with FP8BS_VARIANT_AUTO is the split that runs: the bits of the tiles that have the form, with as many."""
    lib = pkg._lib.load()
    data = _to(pkg.inputs.make_grouped(pkg.inputs.CONFIGS[4], tokens=37, n=518, k=1152, experts=5, topk=2), dev)
    ws = torch.randint(0, 256, (64 << 20,), dtype=torch.uint8, device=dev)
    fresh = lambda: data[:5] + (torch.full_like(data[5], float("nan")),)
    for split in (1, 2, 3, 9):
        want = _grouped_ws(lib, fresh(), 12, split, ws)
        assert torch.equal(_grouped_ws(lib, fresh(), 0, split, ws).view(torch.int16), want.view(torch.int16)), split
