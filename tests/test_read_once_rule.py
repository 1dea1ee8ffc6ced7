"""Which experts' weights a grouped product reads past the caches (fp8bs_kernels.h, `expert_read_once`; fp8bs_tiled.h, `b_read_once`).  Host checks only."""
import ctypes
import os
import subprocess
import sys

import pytest

from test_tall_rows_rule import SHIM

MIB = 1 << 20

# The shim of test_tall_rows_rule.py: each launch prints its kernel's address as the LDS limit is raised.  A limit is raised once a device, so the shim's
# hipGetDevice names another device at each call: without that a kernel's second launch would print nothing.
CALL = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib, one = ctypes.CDLL(sys.argv[2]), ctypes.c_void_p(1 << 20)
for experts, rows, n, k in ((8, 64, 4096, 2048), tuple(map(int, sys.argv[4:]))):
    assert lib.fp8bs_gemm_grouped_ex(one, one, one, one, one, one, experts, rows, n, k, int(sys.argv[3]), None) == 0
    print("-", flush=True)
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "shim.so"), str(d / "shim.c")], check=True)
    return str(d / "shim.so")


def test_by_the_experts_that_have_rows(pkg, tmp_path):
    """Weights that the caches hold are read through them, however many experts the call names; so are those of an expert with a second row of tiles."""
    csrc = os.path.join(os.path.dirname(pkg._lib.LIB_PATH), "csrc")
    (tmp_path / "rule.cpp").write_text("""
#include "fp8bs_kernels.h"
extern "C" int rule(int active, int tile_rows, int n, int k) { return fp8bs::expert_read_once(active, tile_rows, n, k); }
""")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", "-I" + csrc, "-o", str(tmp_path / "rule.so"),
                    str(tmp_path / "rule.cpp")], check=True)
    rule = ctypes.CDLL(str(tmp_path / "rule.so")).rule
    for active, n, k, taken in ((20, 4096, 2048, False), (32, 4096, 2048, False), (35, 4096, 2048, False), (36, 4096, 2048, True), (21, 4096, 7168, True),
                                (2, 1 << 16, (1 << 16) - 128, True), (1, 1 << 16, (1 << 16) - 128, True), (0, 4096, 7168, False)):
        assert bool(rule(active, 1, n, k)) == taken
        assert not rule(active, 2, n, k) and not rule(active, 9, n, k)


# Forced tiles: a call that cannot read 288 MiB of weights, one that can, few rows; rows of b that are no whole lines; the line on the rows an expert.
@pytest.mark.parametrize("tile,experts,rows,n,k,once", [(12, 33, 264, 4096, 2048, False), (12, 36, 288, 4096, 2048, True), (12, 64, 32, 4096, 2048, False), (12, 36, 288, 4160, 2048, False),
                                                        (12, 36, 36 * 48, 4096, 2048, True), (12, 36, 36 * 48 + 4, 4096, 2048, False), (2, 36, 36 * 192, 4096, 2048, True),
                                                        (2, 36, 36 * 192 + 4, 4096, 2048, False), (10 | 2 << 8, 36, 36 * 96, 4096, 2048, True), (10 | 2 << 8, 36, 36 * 96 + 4, 4096, 2048, False)])
def test_the_kernel_of_a_call(pkg, shim, tile, experts, rows, n, k, once):
    out = subprocess.run([sys.executable, "-c", CALL, shim, pkg._lib.LIB_PATH] + [str(v) for v in (tile, experts, rows, n, k)],
                         check=True, stdout=subprocess.PIPE, text=True, timeout=100).stdout
    small, call, _ = out.split("-\n")
    assert small and call and (small != call) == once
