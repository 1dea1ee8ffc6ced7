"""The 128x256 tile: which grouped calls take it, what is refused, and that it keeps its registers.  Host checks only."""
import ctypes

import pytest

from test_kernel_resources import spills  # noqa: F401  (a fixture)
from test_launch_grids import launches, shim  # noqa: F401

ONE = ctypes.c_void_p(16)                                    # never dereferenced
TALL = 10 | 2 << 8                                           # FP8BS_VARIANT_FORM(FP8BS_VARIANT_T256x128S3, 1)
LDS = 3 * (128 + 256) * 128                                  # three stages of a and b, without the scales


# Weights past the 256 MiB line or not, rows an expert at both ends of the rule, 64x256 tiles that fit the chip at once, rounds that are full.
@pytest.mark.parametrize("experts,rows,n,k,taken", [(32, 32 * 16, 4096, 7168, False), (32, 32 * 16 + 1, 4096, 7168, True), (32, 32 * 44, 4096, 7168, True),
                                                    (32, 32 * 44 + 1, 4096, 7168, False), (32, 32 * 64, 3072, 4096, True), (32, 32 * 64 + 1, 3072, 4096, False),
                                                    (32, 1200, 1280, 7168, False), (8, 256, 6144, 7168, False), (8, 384, 6144, 7168, True),
                                                    (32, 32 * 30, 2048, 4096, True), (31, 31 * 30, 2048, 4096, False), (32, 32 * 30, 3000, 4096, False)])
def test_rule(pkg, shim, experts, rows, n, k, taken):  # noqa: F811
    (_, _, _, threads, lds), = launches(pkg, shim, "grouped", experts, rows, n, k)
    assert (threads == 512 and LDS < lds < LDS + 20000) == taken, (threads, lds)


def test_dense_calls_and_splits_are_refused(pkg):
    lib, bad_variant = pkg._lib.load(), 7
    for split in (-1, 0, 1, 2, 2 | pkg._lib.SPLIT_SUM_IN_KERNEL):
        assert lib.fp8bs_gemm_ex(ONE, ONE, ONE, ONE, ONE, ONE, 1 << 40, 256, 512, 1024, TALL, split, None) == bad_variant
    assert lib.fp8bs_gemm_grouped_ws(ONE, ONE, ONE, ONE, ONE, ONE, 4, 64, 256, 1024, TALL, 2, ONE, 1 << 40, None) == bad_variant
    assert pkg._lib.tile_name(TALL) == "t128x256s3"


def test_kernels_do_not_spill(spills):  # noqa: F811
    for mode, epi in ((2, 0), (6, 0), (2, 1), (6, 1)):
        assert spills["128,256,64,64,%d,%d,3,false,false" % (mode, epi)] == 0
