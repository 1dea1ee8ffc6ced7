"""K partitions whose sum is shared out among a tile's workgroups (fp8bs_gemm_ex with split_k | FP8BS_SPLIT_SUM_IN_KERNEL on the
64x64, 64x256 and 128x128 eight-wave tiles, more than eight tiles, all workgroups on the chip at once): the bits of the same
partitions added by the reduce kernel, whatever the workspace holds, also where workgroups give up waiting and leave their part to
another, and where a captured launch takes the sum by one workgroup instead.

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
TILES = (FORM(4, 1), 12, FORM(12, 1))
SHAPES = [(65, 600, 1152), (1, 1200, 1024), (300, 500, 2048), (257, 1030, 1408), (1021, 264, 1536), (640, 512, 1024), (16, 4097, 1152)]


def _operands(pkg, m, n, k, dev):
    return tuple(t.to(dev) for t in pkg.inputs.make_dense(pkg.inputs.CONFIGS[2], m=m, n=n, k=k))


def _check(pkg, dev, shapes):
    flag = pkg._lib.SPLIT_SUM_IN_KERNEL
    ws = importlib.import_module("amd-developer-challenge-2025_amd.submission")._workspace(dev, 64 << 20, torch.cuda.current_stream().cuda_stream)
    for m, n, k in shapes:
        data = _operands(pkg, m, n, k, dev)
        for split in (2, 3, 4, 6, 8):
            if split > k // 128:
                continue
            want = pkg.custom_kernel(data, variant=3, split_k=split).clone()
            for tile in TILES:
                for fill in (0, 255, None):
                    if fill is not None:
                        ws[:16384].fill_(fill)               # (None: as the call before left it)
                    data[4].fill_(float("nan"))
                    out = pkg.custom_kernel(data, variant=tile, split_k=split | flag)
                    assert torch.equal(out.view(torch.int16), want.view(torch.int16)), "%dx%dx%d tile %#x split %d" % (m, n, k, tile, split)


def test_the_bits_of_the_reduce_kernel(pkg):
    _check(pkg, torch.device("cuda:0"), SHAPES)


def test_parts_that_are_left_behind():
    """FP8BS_STREAMK_SPIN < 0: a workgroup looks at the others' flags once, so most leave their part to a later one."""
    env = dict(os.environ, FP8BS_STREAMK_SPIN="-1")
    code = ("import importlib, sys, torch; sys.path[:0] = [%r, %r]; t = importlib.import_module('test_gpu_shared_sum');"
            "t._check(importlib.import_module('amd-developer-challenge-2025_amd'), torch.device('cuda:0'), t.SHAPES); print('all equal')") % (ROOT, os.path.join(ROOT, "tests"))
    res = subprocess.run([sys.executable, "-c", code], env=env, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=110)
    assert res.returncode == 0 and "all equal" in res.stdout, res.stdout[-500:] + res.stderr[-2000:]


@pytest.mark.parametrize("m,n,k,split", [(250, 4096, 7168, 4), (64, 4096, 7168, 8), (300, 500, 2048, 2)])
def test_captured_calls_and_the_epilogue(pkg, m, n, k, split):
    """The planner's own calls: eager, captured and replayed with changed operands, and with the silu-mul epilogue."""
    dev, moe = torch.device("cuda:0"), importlib.import_module("amd-developer-challenge-2025_amd.moe")
    a, b, sa, sb, c = _operands(pkg, m, n, k, dev)
    plan = pkg.plan(m, n, k)
    if split > 2:
        assert plan.split_k == split and not plan.sum_in_kernel      # what a caller with no more than workspace_bytes gets
    want = pkg.custom_kernel((a, b, sa, sb, torch.empty_like(c)), variant=3, split_k=plan.split_k)
    assert torch.equal(pkg.custom_kernel((a, b, sa, sb, c)).view(torch.int16), want.view(torch.int16))
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
