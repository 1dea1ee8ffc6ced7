"""K partitions whose sum is shared out among a tile's workgroups (fp8bs_gemm_ex with split_k | FP8BS_SPLIT_SUM_IN_KERNEL on the
64x64 - from four partitions on -, 64x256 and 128x128 eight-wave tiles, more than eight tiles, all workgroups on the chip at once): the
bits of the same partitions added by the reduce kernel, plain, with the silu-mul epilogue and grouped, whatever the workspace holds, also
where workgroups give up waiting and leave their part to another, and where a captured launch takes another form instead.  That a sum was
shared out shows in the workspace: its flags stay up, where the sum by one workgroup takes its counters down.

The reference merges its K partitions in a second kernel (1-amd-fp8-mm/amd-fp8-mm-submission.py:371-511).
"""
import importlib
import os
import subprocess
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
TILES = ((FORM(4, 1), 64, 64), (12, 64, 256), (FORM(12, 1), 128, 128))
SHAPES = [(65, 600, 1152), (1, 1200, 1024), (300, 500, 2048), (257, 1030, 1408), (1021, 264, 1536), (640, 512, 1024), (16, 4097, 1152)]
GROUPED = [(96, 600, 1152), (75, 1026, 1408)]


def _operands(pkg, m, n, k, dev):
    return tuple(t.to(dev) for t in pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=m, n=n, k=k))


def _shares(tiles, split, tile_n):
    """Can the sums be shared out: two workgroups of 64x64 fit a CU, one of the others."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return tiles > 8 and tiles * split <= cus * (2 if tile_n == 64 else 1) and split >= (4 if tile_n == 64 else 2)


def _flags(ws):
    """The flags that a call left in a workspace whose head was zero: each holds one tag above 1 (stored), 2 (own part left) or 3 (claimed)."""
    words = ws[256:16384].view(torch.int64)
    words = words[words != 0]
    assert len({int(w) >> 16 for w in words}) <= 1
    return [int(w) & 0xFFFF for w in words]


def _check(pkg, dev, shapes):
    """Returns how many parts were left to another workgroup."""
    flag, lib, stream, claimed = pkg._lib.SPLIT_SUM_IN_KERNEL, pkg._lib.load(), torch.cuda.current_stream().cuda_stream, 0
    ws = importlib.import_module("amd-developer-challenge-2025_amd.submission")._workspace(dev, 64 << 20, stream)
    for m, n, k in shapes:
        data = _operands(pkg, m, n, k, dev)
        silu = [torch.empty(m, n // 2, dtype=torch.bfloat16, device=dev) for _ in range(2)]

        def gate_up(out, tile, split):
            assert lib.fp8bs_gemm_silu_mul_ws(*(t.data_ptr() for t in data[:4]), out.data_ptr(), None, 0, m, n, k, tile, split, ws.data_ptr(), ws.numel(), stream) == 0
        for split in (2, 3, 4, 6, 8):
            if split > k // 128:
                continue
            want = pkg.custom_kernel(data, variant=3, split_k=split).clone()
            for tile, tm, tn in TILES:
                tiles = -(-m // tm) * -(-n // tn)
                shared = _shares(tiles, split, tn)
                for fill in (0, 255, None):
                    if fill is not None:
                        ws[:16384].fill_(fill)               # (None: as the call before left it)
                    data[4].fill_(float("nan"))
                    out = pkg.custom_kernel(data, variant=tile, split_k=split | flag)
                    assert torch.equal(out.view(torch.int16), want.view(torch.int16)), "%dx%dx%d tile %#x split %d" % (m, n, k, tile, split)
                    if fill == 0:
                        up = _flags(ws)
                        assert len(up) == (tiles * split if shared else 0) and 2 not in up, "%dx%dx%d tile %#x split %d" % (m, n, k, tile, split)
                        claimed += up.count(3)
                if n % 2 == 0:
                    gate_up(silu[0], tile, split)            # planes, and the epilogue in the reduce kernel
                    silu[1].fill_(float("nan"))
                    ws[:16384].fill_(0)
                    gate_up(silu[1], tile, split | flag)
                    assert torch.equal(silu[0].view(torch.int16), silu[1].view(torch.int16)), "silu-mul %dx%dx%d tile %#x split %d" % (m, n, k, tile, split)
                    up = _flags(ws)
                    assert len(up) == (tiles * split if shared else 0) and 2 not in up
                    claimed += up.count(3)
    return claimed


def _check_grouped(pkg, dev, tokens, n, k):
    """Every expert's rows against the same split of a dense product of them.  Returns how many parts were left to another workgroup."""
    lib, stream, claimed = pkg._lib.load(), torch.cuda.current_stream().cuda_stream, 0
    a, b, sa, sb, ro, c = (t.to(dev) for t in pkg.inputs.make_grouped(pkg.inputs.CONFIGS[4], tokens=tokens, n=n, k=k, experts=4, topk=2))
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
    kmajor = lambda t: t.t().contiguous().t()
    for split in (2, 3, 4, 6):
        rows = ro.tolist()
        want = torch.cat([pkg.custom_kernel((kmajor(a[r0:r1]), b[e], kmajor(sa[r0:r1]), sb[e], torch.empty(r1 - r0, n, dtype=torch.bfloat16, device=dev)), variant=3, split_k=split)
                          for e, (r0, r1) in enumerate(zip(rows, rows[1:])) if r1 > r0])
        for tile, tm, tn in TILES:
            slots = (4 + rows[-1] // (tm - 14)) * -(-n // tn)               # what the launch is sized for
            c.fill_(float("nan"))
            ws[:16384].fill_(0)
            assert lib.fp8bs_gemm_grouped_ws(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr(), ro.data_ptr(), 4, rows[-1], n, k, tile, split,
                                             ws.data_ptr(), ws.numel(), stream) == 0
            assert torch.equal(c.view(torch.int16), want.view(torch.int16)), "grouped %dx%dx%d tile %#x split %d" % (rows[-1], n, k, tile, split)
            up = _flags(ws)
            assert bool(up) == _shares(slots, split, tn) and 2 not in up and len(up) % split == 0
            claimed += up.count(3)
    return claimed


def test_the_bits_of_the_reduce_kernel(pkg):
    _check(pkg, torch.device("cuda:0"), SHAPES)


@pytest.mark.parametrize("tokens,n,k", GROUPED)
def test_the_bits_of_dense_products_of_each_expert(pkg, tokens, n, k):
    _check_grouped(pkg, torch.device("cuda:0"), tokens, n, k)


def test_parts_that_are_left_behind():
    """FP8BS_STREAMK_SPIN < 0: a workgroup looks at the others' flags once, so most leave their part to a later one."""
    env = dict(os.environ, FP8BS_STREAMK_SPIN="-1")
    code = ("import importlib, sys, torch; sys.path[:0] = [%r, %r]; t = importlib.import_module('test_gpu_shared_sum');"
            "p, d = importlib.import_module('amd-developer-challenge-2025_amd'), torch.device('cuda:0');"
            "left = t._check(p, d, t.SHAPES), sum(t._check_grouped(p, d, *g) for g in t.GROUPED); assert min(left) > 0, left; print('all equal', left)") % (ROOT, os.path.join(ROOT, "tests"))
    res = subprocess.run([sys.executable, "-c", code], env=env, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=110)
    assert res.returncode == 0 and "all equal" in res.stdout, res.stdout[-500:] + res.stderr[-2000:]


@pytest.mark.parametrize("m,n,k,split", [(250, 4096, 7168, 4), (64, 4096, 7168, 8), (1024, 1536, 7168, 2), (64, 18432, 7168, 3), (21, 778, 5888, 8)])
def test_captured_calls_and_the_epilogue(pkg, m, n, k, split):
    """The planner's own calls: eager, shared out; captured and replayed with changed operands, not shared; and with the silu-mul epilogue."""
    dev, moe = torch.device("cuda:0"), importlib.import_module("amd-developer-challenge-2025_amd.moe")
    a, b, sa, sb, c = _operands(pkg, m, n, k, dev)
    plan = pkg.plan(m, n, k)
    assert plan.split_k == split and plan.sum_in_kernel == (split in (2, 3))      # what a captured call gets
    want = pkg.custom_kernel((a, b, sa, sb, torch.empty_like(c)), variant=3, split_k=plan.split_k)
    ws = importlib.import_module("amd-developer-challenge-2025_amd.submission")._workspace(dev, 64 << 20, torch.cuda.current_stream().cuda_stream)
    ws[:16384].fill_(0)
    assert torch.equal(pkg.custom_kernel((a, b, sa, sb, c)).view(torch.int16), want.view(torch.int16))
    assert len(_flags(ws)) == plan.grid_x
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pkg.custom_kernel((a, b, sa, sb, c))
    for scale in (1.0, 2.0, 0.5):
        sa.mul_(scale)
        c.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        want = pkg.custom_kernel((a, b, sa, sb, torch.empty_like(c)), variant=3, split_k=plan.split_k)
        assert torch.equal(c.view(torch.int16), want.view(torch.int16))
    h = moe.gate_up_silu((a, b, sa, sb, None, torch.empty(m, n // 2, dtype=torch.bfloat16, device=dev)))
    g = want.float()
    ref = torch.nn.functional.silu(g[:, 0::2]) * g[:, 1::2]
    assert bool(((h.float() - ref).abs() <= 1e-3 + 2 * 2e-2 * ref.abs()).all())


def test_capture_after_one_eager_call_in_a_fresh_process():
    """Four partitions, shared out when eager and in two launches when captured, by a process that has launched nothing else."""
    code = """import importlib, sys, torch
sys.path.insert(0, %r)
pkg = importlib.import_module('amd-developer-challenge-2025_amd')
a, b, sa, sb, c = (t.to('cuda:0') for t in pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=250, n=4096, k=7168))
want = pkg.custom_kernel((a, b, sa, sb, torch.empty_like(c))).clone()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    pkg.custom_kernel((a, b, sa, sb, c))
for _ in range(3):
    c.fill_(3.0)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(c.view(torch.int16), want.view(torch.int16))
print('all equal')""" % ROOT
    res = subprocess.run([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=110)
    assert res.returncode == 0 and "all equal" in res.stdout, res.stdout[-500:] + res.stderr[-2000:]
