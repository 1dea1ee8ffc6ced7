"""Launches of very tall matrices stay inside the documented grid limit of 65535 in y and still cover every row; which of two
kernels a call of the routing functions takes.

On the CPU the launches are recorded instead of made: a small library loaded ahead of the HIP runtime takes the launch
configuration that hipcc's host code hands over, and declines.  No pointer is dereferenced."""
import importlib
import json
import subprocess
import sys

import pytest
import torch

SHIM = r"""
#include <stdint.h>
#include <stdio.h>
typedef struct { uint32_t x, y, z; } grid3;
int __hipPushCallConfiguration(grid3 g, grid3 b, size_t lds, void* stream) {
    (void)stream;
    printf("[%u, %u, %u, %u, %zu]\n", g.x, g.y, g.z, b.x, lds); fflush(stdout);
    return 1;
}
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* f, int attr, int value) { (void)f; (void)attr; (void)value; return 0; }
"""
CALL = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
one = ctypes.c_void_p(1 << 20)
fn, dtype, gathered, rows, k = sys.argv[3], int(sys.argv[4]), int(sys.argv[5]), int(sys.argv[6]), int(sys.argv[7])
if fn == "a":
    st = lib.fp8bs_quantize_a(one, dtype, ctypes.c_int64(k), one if gathered else None, 1000 if gathered else rows, one, one, rows, k, None)
elif fn == "b":
    st = lib.fp8bs_quantize_b(one, dtype, ctypes.c_int64(k), one, one, rows, k, None)
elif fn == "grouped":
    experts, rows, n, k = dtype, gathered, rows, k
    st = lib.fp8bs_gemm_grouped(one, one, one, one, one, one, experts, rows, n, k, None)
elif fn == "combine":
    tokens, topk, d = dtype, gathered, rows
    st = lib.fp8bs_moe_combine(one, tokens * topk, one, one, one, tokens, topk, d, None)
else:
    tokens, experts, topk = dtype, gathered, rows
    st = lib.fp8bs_moe_route(one, tokens, experts, topk, one, one, one, one, ctypes.c_size_t(1 << 30), None)
assert st == 0, st
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "shim.so"), str(d / "shim.c")], check=True)
    return str(d / "shim.so")


def launches(pkg, shim, *args):
    out = subprocess.run([sys.executable, "-c", CALL, shim, pkg._lib.LIB_PATH] + [str(a) for a in args],
                         check=True, stdout=subprocess.PIPE, text=True, timeout=100).stdout
    return [json.loads(line)[:5 if args[0] == "grouped" else 4] for line in out.splitlines()]


@pytest.mark.parametrize("fn,dtype,gathered,rows,k", [("a", 1, 1, 65535 * 32, 128), ("a", 1, 1, 65535 * 32 + 1, 128), ("a", 1, 1, 16000001, 256), ("a", 0, 0, 65535 * 64 + 1, 128),
                                                      ("a", 0, 0, 8388607, 128), ("a", 1, 0, 16777215, 128), ("b", 1, 0, 65535 * 128, 128), ("b", 1, 0, 65535 * 128 + 1, 128),
                                                      ("a", 1, 0, 300, 256), ("b", 0, 0, 129, 128)])
def test_rows_beyond_the_grid_limit(pkg, shim, fn, dtype, gathered, rows, k):
    grids = launches(pkg, shim, fn, dtype, gathered, rows, k)
    assert grids and all(g[0] == k // 128 and 1 <= g[1] <= 65535 and g[2] == 1 and g[3] == 256 for g in grids), grids
    assert sum(g[1] for g in grids) in [-(-rows // r) for r in ((128,) if fn == "b" else (32, 64, 128))]


@pytest.mark.parametrize("tokens,experts,topk,one", [(256, 1024, 16, True), (1024, 32, 7, True), (900, 32, 8, True), (512, 256, 7, True), (700, 128, 7, True),
                                                      (1024, 256, 2, True), (1024, 256, 7, False), (1024, 128, 7, False), (900, 128, 8, False),
                                                      (700, 256, 8, False), (1024, 32, 8, False), (1025, 8, 1, False)])
def test_routing_in_one_workgroup_where_that_is_faster(pkg, shim, tokens, experts, topk, one):
    """Many rows to many experts leave one workgroup slower than two kernels over several."""
    threads = [g[3] for g in launches(pkg, shim, "route", tokens, experts, topk, 0)]
    assert threads == ([256, 256] if not one else [256] if tokens <= 256 else [1024])


@pytest.mark.parametrize("tokens,topk,d,split", [(1, 8, 7168, True), (768, 1, 7168, True), (1024, 8, 7168, True), (1024, 6, 5120, True), (64, 8, 2056, True),
                                                 (1024, 1, 7168, False), (1000, 2, 7168, False), (1024, 4, 4096, False), (1025, 8, 7168, False), (64, 8, 2048, False)])
def test_combining_over_several_workgroups_where_that_is_faster(pkg, shim, tokens, topk, d, split):
    assert launches(pkg, shim, "combine", tokens, topk, d, 0) == ([[tokens, -(-d // 1024), 1, 128]] if split else [[tokens, 1, 1, 256]])


@pytest.mark.parametrize("dtype,t,m,k,aligned,two", [
    (torch.bfloat16, 4096, 32768, 7168, True, True), (torch.bfloat16, 4096, 20480, 7168, True, True), (torch.bfloat16, 2048, 16384, 7168, True, True),
    (torch.bfloat16, 6016, 48128, 4096, True, True), (torch.bfloat16, 6016, 36096, 4096, True, False), (torch.bfloat16, 6976, 55808, 7168, True, False),
    (torch.float32, 6016, 24064, 4096, True, True), (torch.bfloat16, 4096, 16384, 7168, True, False), (torch.bfloat16, 4096, 20480, 4096, True, False), (torch.bfloat16, 8192, 65536, 2048, True, False),
    (torch.bfloat16, 16384, 131072, 1024, True, False), (torch.bfloat16, 4094, 32752, 7168, True, False), (torch.bfloat16, 4096, 32768, 7168, False, False),
    (torch.float32, 4096, 16384, 7168, True, True), (torch.float32, 4096, 16384, 4096, True, True), (torch.float32, 2048, 8192, 7168, True, True),
    (torch.float32, 1024, 8192, 7168, True, True), (torch.float32, 8192, 40960, 4096, True, True), (torch.float32, 4096, 8192, 7168, True, False),
    (torch.float32, 8192, 65536, 1024, True, False), (torch.float32, 16384, 131072, 2048, True, False)])
def test_the_faster_route_of_a_gathered_quantisation(monkeypatch, dtype, t, m, k, aligned, two):
    """One kernel that gathers as it quantises, or two: shapes where each is faster by measurement.  The calls stop before the library's."""
    quant = importlib.import_module("amd-developer-challenge-2025_amd.quant")
    calls = []
    monkeypatch.setattr(quant, "_check_input", lambda x, name: None)
    monkeypatch.setattr(quant, "_call", lambda fn, *args: calls.append("quantise"))
    monkeypatch.setattr(quant, "gather_a", lambda *args: calls.append("gather"))
    monkeypatch.setattr(quant, "_k_major", lambda rows, k, dtype, device: torch.empty(0, device="cpu"))
    x = torch.empty(t, 1, dtype=dtype).expand(t, k)                # sizes and addresses are all that is looked at
    row_map = torch.empty(m + 8, dtype=torch.int32)
    row_map = row_map[-row_map.data_ptr() % 16 // 4 + (0 if aligned else 1):][:m]
    quant.quantize_a(x, row_map)
    assert calls == (["quantise", "gather"] if two else ["quantise"])


@pytest.mark.parametrize("tokens,experts,topk,n,k,tile", [(640, 32, 4, 3664, 5376, 2), (704, 32, 8, 2176, 1280, 2), (931, 16, 8, 3806, 5888, 2), (2972, 16, 2, 3200, 1408, 2),
                                                          (4096, 32, 8, 4096, 7168, 2), (704, 16, 4, 512, 1280, 12 | 2 << 8), (32, 32, 8, 4096, 7168, 12)])
def test_the_tile_of_a_grouped_call(pkg, shim, tokens, experts, topk, n, k, tile):
    """Shapes on which the tile is the fastest by measurement, known here by its threads and its LDS."""
    (_, _, _, threads, lds), = launches(pkg, shim, "grouped", experts, tokens * topk, n, k)
    assert threads == 512 and lds == {2: 2 * (128 * 512 + 1024 + 256), 12: 3 * (128 * 320 + 1024 + 256), 12 | 2 << 8: 4 * (128 * 256 + 1024 + 256)}[tile]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows", [("gathered", 65535 * 32 + 33), ("f32", 65535 * 64 + 70), ("b", 65535 * 128 + 200)])
def test_values_on_both_sides_of_the_grid_limit(kind, rows):
    """The rows of the second launch: the bytes and scales of the same rows quantised on their own."""
    quant = importlib.import_module("amd-developer-challenge-2025_amd.quant")
    dev = torch.device("cuda:0")
    base = torch.randn(1024, 128, generator=torch.Generator().manual_seed(3)) * torch.logspace(-3, 3, 1024)[:, None]
    base = base.to(torch.float32 if kind == "f32" else torch.bfloat16).to(dev)
    if kind == "gathered":
        rmap = (torch.arange(rows, dtype=torch.int64, device=dev) * 7 % 1024).to(torch.int32)
        q, s = quant.quantize_a(base, rmap, fused=True)
    else:
        rmap = torch.arange(rows, device=dev) % 1024
        q, s = (quant.quantize_b if kind == "b" else quant.quantize_a)(base.repeat(-(-rows // 1024), 1)[:rows])
    at = rmap.long()
    if kind == "b":
        wq, ws = quant.quantize_b(base)
        whole = rows // 128                                                    # (the last block has other rows, and may have another maximum)
        assert torch.equal(s[:whole, 0], ws[torch.arange(whole, device=dev) % 8, 0])
        rows = whole * 128
    else:
        wq, ws = quant.quantize_a(base)
        assert torch.equal(s[:, 0], ws[:, 0][at])
    assert torch.equal(q.t()[:, :rows].view(torch.uint8), wq.t().view(torch.uint8)[:, at[:rows]])
