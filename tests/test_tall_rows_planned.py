"""Which grouped calls with a workspace take the 128x256 tile: by the rounds that 64x256 tiles take, in the place of a K split, and not.  Host checks only."""
import subprocess
import sys

import pytest

from test_tall_rows_rule import SHIM, TALL

# Each launch prints its kernel's address as the LDS limit is raised.  A limit is raised once a device, so the shim's hipGetDevice names another device at each
# call: without that a kernel's second launch would print nothing.
CALL = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib, one = ctypes.CDLL(sys.argv[2]), ctypes.c_void_p(1 << 20)
experts, rows, n, k, tall = map(int, sys.argv[3:])
assert lib.fp8bs_gemm_grouped_ws(one, one, one, one, one, one, experts, rows, n, k, 0, 0, one, ctypes.c_size_t(1 << 40), None) == 0
print("-", flush=True)
assert lib.fp8bs_gemm_grouped_ws(one, one, one, one, one, one, experts, rows, n, k, tall, 1, None, ctypes.c_size_t(0), None) == 0
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "shim.so"), str(d / "shim.c")], check=True)
    return str(d / "shim.so")


# Up to 44 rows an expert: 64x256 tiles whose second rows fit the last round keep the call, those that start another and other tiles do not; calls that were
# split, by either rule; one that still is.
@pytest.mark.parametrize("experts,rows,n,k,taken,splits", [(32, 1300, 4736, 3072, False, False), (16, 529, 4864, 3456, False, False), (64, 1194, 1664, 4480, False, False),
                                                           (32, 727, 4096, 3712, True, False), (32, 1350, 3200, 5760, True, False), (64, 2698, 5120, 1920, True, False),
                                                           (32, 1191, 2176, 5248, True, False), (16, 1699, 2139, 5888, True, False), (16, 512, 1024, 7168, False, True)])
def test_calls_with_a_workspace(pkg, shim, experts, rows, n, k, taken, splits):
    out = subprocess.run([sys.executable, "-c", CALL, shim, pkg._lib.LIB_PATH] + [str(v) for v in (experts, rows, n, k, TALL)],
                         check=True, stdout=subprocess.PIPE, text=True, timeout=100).stdout
    planned, forced = out.split("-\n")
    assert planned and forced and (planned == forced) == taken
    assert (pkg._lib.load().fp8bs_grouped_workspace_bytes(experts, rows, n, k) > 0) == splits
