"""What a call launches when its stream is captured, and what an eager call of the same shape has made ready for it.

On the CPU: a small library loaded ahead of the HIP runtime says whether the stream is capturing, and takes the launches and the
attribute calls instead of the runtime.  No pointer is dereferenced."""
import json
import subprocess
import sys

import pytest

SHIM = r"""
#include <stdint.h>
#include <stdio.h>
typedef struct { uint32_t x, y, z; } grid3;
static int capturing;
static grid3 g_, b_; static size_t lds_;
void shim_capture(int on) { capturing = on; }
int hipStreamIsCapturing(void* stream, int* status) { (void)stream; *status = capturing; return 0; }
int __hipPushCallConfiguration(grid3 g, grid3 b, size_t lds, void* stream) { (void)stream; g_ = g; b_ = b; lds_ = lds; return 0; }
int __hipPopCallConfiguration(grid3* g, grid3* b, size_t* lds, void** stream) { *g = g_; *b = b_; *lds = lds_; *stream = 0; return 0; }
int hipLaunchKernel(const void* f, grid3 g, grid3 b, void** args, size_t lds, void* stream) {
    (void)args; (void)stream;
    printf("{\"launch\": %zu, \"grid\": %u, \"threads\": %u, \"lds\": %zu}\n", (size_t)f, g.x, b.x, lds); fflush(stdout);
    return 0;
}
int hipGetLastError(void) { return 0; }
int hipGetDevice(int* device) { *device = 0; return 0; }
int hipDeviceGetAttribute(int* value, int attr, int device) { (void)attr; (void)device; *value = 256; return 0; }       /* CUs */
int hipFuncSetAttribute(const void* f, int attr, int value) { (void)attr; (void)value; printf("{\"raise\": %zu}\n", (size_t)f); fflush(stdout); return 0; }
"""
CALLS = r"""
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
one = ctypes.c_void_p(1 << 20)
for fn, capture, m, n, k, variant, split, ws_bytes in json.loads(sys.argv[3]):
    shim.shim_capture(capture)
    print(json.dumps({"call": [fn, capture, m, n, k, variant, split]}), flush=True)
    ws = (one, ctypes.c_size_t(ws_bytes)) if ws_bytes else (None, ctypes.c_size_t(0))
    if fn == "gemm":
        st = lib.fp8bs_gemm_ex(one, one, one, one, one, *ws, m, n, k, variant, split, None)
    elif fn == "silu":
        st = lib.fp8bs_gemm_silu_mul_ws(one, one, one, one, one, None, 0, m, n, k, variant, split, *ws, None)
    else:
        st = lib.fp8bs_gemm_grouped_ws(one, one, one, one, one, one, 4, m, n, k, variant, split, *ws, None)
    assert st == 0, st
"""
FORM = lambda variant, form: variant | (form + 1) << 8           # FP8BS_VARIANT_FORM
SUM = 1 << 30                                                    # FP8BS_SPLIT_SUM_IN_KERNEL
MUCH = 256 << 20


@pytest.fixture(scope="module")
def run(pkg, tmp_path_factory):
    """run(calls): for every call ("gemm" | "silu" | "grouped", capturing, m, n, k, variant, split, workspace bytes) in one fresh
    process, the list of what it launched and the list of the kernels whose LDS limit it raised."""
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "shim.so"), str(d / "shim.c")], check=True)

    def call(calls):
        out = subprocess.run([sys.executable, "-c", CALLS, str(d / "shim.so"), pkg._lib.LIB_PATH, json.dumps(calls)],
                             check=True, stdout=subprocess.PIPE, text=True, timeout=100).stdout
        seen = []
        for line in map(json.loads, out.splitlines()):
            if "call" in line:
                seen.append(([], []))
            elif "launch" in line:
                seen[-1][0].append(line)
            else:
                seen[-1][1].append(line["raise"])
        assert len(seen) == len(calls)
        return seen
    return call


@pytest.mark.parametrize("fn,variant,m,n,k,split", [("gemm", FORM(4, 1), 448, 924, 4480, 4), ("gemm", 12, 64, 18432, 7168, 3), ("gemm", FORM(12, 1), 1876, 571, 4608, 3),
                                                    ("gemm", FORM(12, 1), 250, 4096, 7168, 4), ("silu", FORM(12, 1), 250, 4096, 7168, 2), ("grouped", FORM(4, 1), 96, 832, 1024, 4)])
def test_a_captured_sum_has_a_kernel_without_the_shared_one(run, fn, variant, m, n, k, split):
    """A captured launch cannot share out its sums.  Its kernel is the one that an eager call takes where there is nothing to
    share (eight tiles and fewer), not one that carries both forms and is the slower for it."""
    few = (fn, 0, 16, 66 if m % 4 or n % 8 else 64, k, variant, split | SUM, MUCH)              # (rows as whole or as odd: the same instantiation)
    (eager, _), (captured, raised), (small, _) = run([(fn, capture, m, n, k, variant, split | SUM, MUCH) for capture in (0, 1)] + [few])
    assert len(eager) == len(captured) == len(small) == 1
    assert not raised                                                 # the eager call has readied the captured one's kernel
    assert eager[0]["launch"] != captured[0]["launch"]
    assert (eager[0]["grid"], eager[0]["threads"], eager[0]["lds"]) == (captured[0]["grid"], captured[0]["threads"], captured[0]["lds"])
    assert captured[0]["launch"] == small[0]["launch"]


@pytest.mark.parametrize("fn,m,n,k", [("gemm", 192, 1280, 3072), ("gemm", 448, 512, 3456), ("silu", 128, 1472, 2304), ("grouped", 96, 832, 1024)])
def test_two_or_three_partitions_of_64x64_are_not_shared(run, fn, m, n, k):
    """Four accumulators a wave in three parts: the shared sum is slower than the sum by one workgroup, which is what runs."""
    calls = [(fn, capture, m, n, k, FORM(4, 1), split | SUM, MUCH) for split in (2, 3, 4) for capture in (0, 1)]
    kernels = [launched[0]["launch"] for launched, _ in run(calls)]
    assert kernels[0] == kernels[1] == kernels[2] == kernels[3] == kernels[5] != kernels[4]


@pytest.mark.parametrize("m,n,k,tile,split", [(896, 1344, 2944, (64, 128), 1), (576, 2048, 3328, (64, 128), 1), (960, 640, 7040, (64, 128), 3), (256, 3648, 4736, (64, 64), 1),
                                              (384, 2637, 6528, (128, 128), 3), (250, 4096, 7168, (128, 128), 4), (64, 4096, 7168, (128, 128), 8), (64, 18432, 7168, (64, 256), 3)])
def test_one_plan_that_is_sound_for_every_caller(pkg, run, m, n, k, tile, split):
    """The same tile and split eager and captured, so that a replay has the bits of an eager call; and not one that is picked at the price of
    a shared sum and takes 4 to 40 % longer without (the first five, before their plans were priced in both forms)."""
    p = pkg.plan(m, n, k)
    assert ((p.tile_m, p.tile_n), p.split_k) == (tile, split)
    (eager, _), (captured, _), (tight, _) = run([("gemm", 0, m, n, k, 0, 0, MUCH), ("gemm", 1, m, n, k, 0, 0, MUCH), ("gemm", 0, m, n, k, 0, 0, int(p.workspace_bytes))])
    for launched in (eager, captured, tight):
        assert (launched[0]["grid"], launched[0]["threads"], launched[0]["lds"]) == (p.grid_x, p.block_threads, p.lds_bytes)
    assert len(captured) == (2 if split > 1 and not p.sum_in_kernel else 1)
    assert len(eager) == 1 and len(tight) == len(captured)


@pytest.mark.parametrize("fn,m,n,k", [("gemm", 250, 4096, 7168), ("silu", 250, 4096, 7168), ("gemm", 64, 4096, 7168), ("gemm", 448, 1537, 5120), ("gemm", 1024, 1536, 7168),
                                      ("gemm", 256, 512, 1024), ("gemm", 64, 512, 7168), ("grouped", 96, 832, 7168)])
def test_one_eager_call_readies_a_capture(run, fn, m, n, k):
    """In a process that has launched nothing else: whatever kernel a captured call of the shape takes, an eager call with the same
    arguments has raised its LDS limit, which is no thing to be done under capture."""
    (eager, _), (captured, raised) = run([(fn, capture, m, n, k, 0, 0, MUCH) for capture in (0, 1)])
    assert eager and captured and not raised


@pytest.mark.parametrize("fn,m,n,k", [("gemm", 250, 4096, 7168), ("gemm", 64, 4096, 7168), ("gemm", 64, 7168, 7168), ("gemm", 448, 1537, 5120), ("silu", 250, 4096, 7168)])
def test_a_workspace_of_the_reported_size_lets_a_sum_be_shared(pkg, run, fn, m, n, k):
    """What fp8bs_workspace_bytes and fp8bs_silu_mul_workspace_bytes say is room for the fastest form, one launch, and for a capture's
    two; a byte less is not, and takes the same split in two."""
    nbytes = pkg._lib.load().fp8bs_silu_mul_workspace_bytes(m, n, k) if fn == "silu" else pkg.workspace_bytes(m, n, k)
    assert nbytes >= pkg.plan(m, n, k).workspace_bytes
    counts = [len(launched) for launched, _ in run([(fn, 0, m, n, k, 0, 0, nbytes), (fn, 1, m, n, k, 0, 0, nbytes), (fn, 0, m, n, k, 0, 0, nbytes - 1)])]
    assert counts == [1, 2, 2]


@pytest.mark.parametrize("m,n,k,split", [(7, 1516, 7040, 8), (14, 3373, 6144, 4), (1, 827, 6656, 8), (11, 2882, 5120, 4), (21, 777, 5888, 8), (46, 2489, 4736, 6),
                                        (41, 1280, 3456, 8), (16, 2096, 3712, 6)])
def test_a_few_rows_share_their_sums(pkg, run, m, n, k, split):
    """One launch of 64x64 tiles: with planes and a reduce launch 10 to 26 % slower where n is odd, and one launch more where it is not."""
    p = pkg.plan(m, n, k)
    assert (p.tile_m, p.tile_n, p.split_k) == (64, 64, split)
    (eager, _), = run([("gemm", 0, m, n, k, 0, 0, pkg.workspace_bytes(m, n, k))])
    assert len(eager) == 1
