"""Which grouped products change a workgroup's columns from round to round (fp8bs_kernels.h, `turns_rounds`).  Host check only."""
import ctypes
import os
import subprocess


def test_by_the_distance_of_rows_of_b(pkg, tmp_path):
    """Where columns fall on the slow bytes of a line of 1024: with rows a multiple of 512 apart, and not where they drift through all of them."""
    csrc = os.path.join(os.path.dirname(pkg._lib.LIB_PATH), "csrc")
    (tmp_path / "rule.cpp").write_text('#include "fp8bs_kernels.h"\nextern "C" int rule(int n) { return fp8bs::turns_rounds(n); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", "-I" + csrc, "-o", str(tmp_path / "rule.so"),
                    str(tmp_path / "rule.cpp")], check=True)
    rule = ctypes.CDLL(str(tmp_path / "rule.so")).rule
    assert all(rule(n) for n in (512, 3584, 4096, 4608, 7168)) and not any(rule(n) for n in (1, 2176, 3001, 4000, 4224, 4352, 4480, 5000))
