"""What the compiler made of the kernels: no instantiation that carries an unsplit product keeps anything in scratch memory, which no count of spilled registers shows."""
import subprocess

import pytest

pytest.importorskip("msgpack")
from test_kernel_resources import TILES, _gfx950_objects, _kernels

READ_ONCE = ["64,256,32,64,6,%d,3", "128,256,64,64,6,%d,3", "256,256,64,128,6,%d,2"]


@pytest.fixture(scope="module")
def kernels(pkg):
    """gemm_tr_kernel's template arguments -> the metadata of the kernel."""
    with open(pkg._lib.LIB_PATH, "rb") as f:
        data = f.read()
    found = {k[".name"]: k for elf in _gfx950_objects(data) for k in _kernels(elf)}
    names = subprocess.run(["c++filt"] + list(found), check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()
    return {n.split("<")[1].split(">")[0].replace(" ", ""): v for n, v in zip(names, found.values()) if "gemm_tr_kernel<" in n}


@pytest.mark.parametrize("tails", ["false", "true"])
@pytest.mark.parametrize("tile", TILES)
def test_dense_and_grouped(kernels, tile, tails):
    if tile.startswith("256,192") and tails == "true":
        pytest.skip("256 registers are not enough for it")
    for mode in (0, 2):
        assert kernels[tile % (mode, 0) + ",%s,false" % tails][".private_segment_fixed_size"] == 0


@pytest.mark.parametrize("tails", ["false", "true"])
@pytest.mark.parametrize("tile", READ_ONCE)
def test_weights_past_the_caches(kernels, tile, tails):
    for epi in (0, 1):
        assert kernels[tile % epi + ",%s,false" % tails][".private_segment_fixed_size"] == 0


@pytest.mark.parametrize("tile", READ_ONCE)
def test_weights_past_the_caches_without_spills(kernels, tile):
    """As the instantiations that they stand in for: aligned operands, plain and with the epilogue."""
    for epi in (0, 1):
        assert kernels[tile % epi + ",false,false"][".vgpr_spill_count"] == 0
