"""The 128x256 tile: which grouped calls take it, what is refused, and that it keeps its registers.  Host checks only."""
import ctypes
import subprocess
import sys

import pytest

from test_kernel_resources import spills  # noqa: F401  (a fixture)

ONE = ctypes.c_void_p(16)                                    # never dereferenced
TALL = 10 | 2 << 8                                           # FP8BS_VARIANT_FORM(FP8BS_VARIANT_T256x128S3, 1)

# Loaded ahead of the HIP runtime: the kernels' addresses are recorded as their LDS limits are raised, every launch is declined.
SHIM = r"""
#include <stdio.h>
typedef struct { unsigned x, y, z; } grid3;
int __hipPushCallConfiguration(grid3 g, grid3 b, size_t lds, void* stream) { (void)g; (void)b; (void)lds; (void)stream; return 1; }
int hipGetLastError(void) { return 0; }
int hipGetDevice(int* device) { static int next = 0; *device = next++ % 8; return 0; }
int hipFuncSetAttribute(const void* f, int attr, int value) { (void)attr; (void)value; printf("%p\n", f); fflush(stdout); return 0; }
"""
CALL = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib, one = ctypes.CDLL(sys.argv[2]), ctypes.c_void_p(1 << 20)
experts, rows, n, k, tall = map(int, sys.argv[3:])
for variant in (0, tall):
    assert lib.fp8bs_gemm_grouped_ex(one, one, one, one, one, one, experts, rows, n, k, variant, None) == 0
    print("-", flush=True)
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "shim.so"), str(d / "shim.c")], check=True)
    return str(d / "shim.so")


# Weights past the 256 MiB line or not, rows an expert at both ends of the rules, 64x256 tiles that fit the chip at once, rounds that are full;
# smaller weights, by the model.
@pytest.mark.parametrize("experts,rows,n,k,taken", [(32, 32 * 16, 4096, 7168, False), (32, 32 * 16 + 1, 4096, 7168, True), (32, 32 * 44, 4096, 7168, True),
                                                    (32, 32 * 44 + 1, 4096, 7168, False), (32, 32 * 64, 3072, 4096, True), (32, 32 * 128 + 1, 3072, 4096, False),
                                                    (32, 32 * 80, 1408, 2048, True), (32, 32 * 44, 1408, 2048, False), (32, 32 * 80, 256, 2048, False),
                                                    (32, 1200, 1280, 7168, False), (8, 256, 6144, 7168, False), (8, 384, 6144, 7168, True),
                                                    (32, 32 * 30, 2048, 4096, True), (31, 31 * 30, 2048, 4096, False), (32, 32 * 30, 3000, 4096, False)])
def test_rule(pkg, shim, experts, rows, n, k, taken):
    out = subprocess.run([sys.executable, "-c", CALL, shim, pkg._lib.LIB_PATH] + [str(v) for v in (experts, rows, n, k, TALL)],
                         check=True, stdout=subprocess.PIPE, text=True, timeout=100).stdout
    planned, forced, _ = out.split("-\n")
    print(out)
    assert forced and (planned == forced) == taken


def test_dense_calls_and_splits_are_refused(pkg):
    lib, bad_variant = pkg._lib.load(), 7
    for split in (-1, 0, 1, 2, 2 | pkg._lib.SPLIT_SUM_IN_KERNEL):
        assert lib.fp8bs_gemm_ex(ONE, ONE, ONE, ONE, ONE, ONE, 1 << 40, 256, 512, 1024, TALL, split, None) == bad_variant
    assert lib.fp8bs_gemm_grouped_ws(ONE, ONE, ONE, ONE, ONE, ONE, 4, 64, 256, 1024, TALL, 2, ONE, 1 << 40, None) == bad_variant
    assert pkg._lib.tile_name(TALL) == "t128x256s3"


def test_kernels_do_not_spill(spills):  # noqa: F811
    for mode, epi in ((2, 0), (6, 0), (2, 1), (6, 1)):
        assert spills["128,256,64,64,%d,%d,3,false,false" % (mode, epi)] == 0
