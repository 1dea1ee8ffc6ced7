"""Plans and forced arguments that name one of the two forms of a variant, or a K split: honoured or refused, never
something else run in their place.  Host checks only: every call here returns before a launch."""
import ctypes
import types
import warnings

import pytest

ONE = ctypes.c_void_p(16)                                    # never dereferenced
FORM = lambda variant, form: variant | (form + 1) << 8      # FP8BS_VARIANT_FORM
BAD_VARIANT, WORKSPACE = 7, 3


def test_dealt_k_blocks_are_refused_for_a_second_form(pkg):
    """split_k < 0 deals K blocks, which the second forms do not have; the first forms get as far as the workspace check."""
    lib = pkg._lib.load()
    for variant in (4, 12):
        assert lib.fp8bs_gemm_ex(ONE, ONE, ONE, ONE, ONE, None, 0, 256, 512, 1024, FORM(variant, 1), -1, None) == BAD_VARIANT
        assert lib.fp8bs_gemm_ex(ONE, ONE, ONE, ONE, ONE, None, 0, 256, 512, 1024, FORM(variant, 0), -1, None) == WORKSPACE
        assert lib.fp8bs_gemm_ex(ONE, ONE, ONE, ONE, ONE, None, 0, 256, 512, 1024, variant, -1, None) == WORKSPACE


def test_a_plan_is_run_again_and_named_with_its_form(pkg):
    """The variant alone names its first form: another tile, with another name and another workspace need."""
    lib, second = pkg._lib.load(), 0
    for m, n, k in [(512, 2048, 1024), (1024, 1536, 7168), (2048, 1152, 4096), (640, 1536, 7168), (64, 18432, 7168), (4096, 4096, 4096), (4096, 2112, 7168)]:
        p = pkg.plan(m, n, k)
        again = pkg._lib.planned_variant(p)
        assert "%dx%d" % (p.tile_m, p.tile_n) in pkg._lib.tile_name(again)
        second += p.form
        if p.sum_in_kernel:
            split = p.split_k | pkg._lib.SPLIT_SUM_IN_KERNEL
            assert lib.fp8bs_gemm_ex(ONE, ONE, ONE, ONE, ONE, ONE, p.workspace_bytes - 4, m, n, k, again, split, None) == WORKSPACE
    assert second >= 2
    assert [pkg._lib.tile_name(v) for v in (0, 2, 12, FORM(12, 0), FORM(12, 1), 4, FORM(4, 1))] == ["auto", "t256x256", "t64x256s3", "t64x256s3", "t128x128s4", "t64x128", "t64x64s4"]
    assert lib.fp8bs_version() >= 400


def test_a_forced_grouped_split_is_honoured_or_refused(pkg):
    """Also with the tile left to the library, as in a dense call: a split that cannot be done, or not with this workspace,
    is an error and not another split."""
    lib = pkg._lib.load()
    for fn in (lib.fp8bs_gemm_grouped_ws, lib.fp8bs_gemm_silu_mul_ws):
        call = lambda variant, split, k=1024: fn(ONE, ONE, ONE, ONE, ONE, ONE, 4, 64, 256, k, variant, split, None, 0, None)
        for variant in (0, 12, FORM(4, 1)):
            assert call(variant, 2) == WORKSPACE and call(variant, 2 | pkg._lib.SPLIT_SUM_IN_KERNEL) == WORKSPACE
            assert call(variant, 9) == BAD_VARIANT                          # more partitions than K blocks
            assert call(variant, -1) == BAD_VARIANT
        assert call(2, 2) == BAD_VARIANT                                    # a tile without the form


def test_long_chains_take_the_tile_that_measures_fastest(pkg):
    """Chains of 49 to 80 K blocks in about one round of 128x128 tiles: eight waves, unsplit (5 to 12 % faster on MI355X than
    the best of the other tiles); beyond 80 the split 256x128 tile is ahead."""
    for m, n, k in [(6144, 512, 7168), (2048, 2048, 7168), (4096, 1024, 7168), (1536, 2304, 7168), (1024, 3072, 7168), (4096, 768, 7168),
                    (2048, 1536, 7168), (4096, 1024, 6272), (3072, 1280, 7168), (2048, 2048, 10240)]:
        p = pkg.plan(m, n, k)
        assert (p.variant, p.form, p.split_k) == (12, 1, 1), (m, n, k)
    for m, n, k in [(2048, 2048, 14336), (4096, 1024, 16384)]:
        p = pkg.plan(m, n, k)
        assert (p.tile_m, p.tile_n, p.split_k, p.sum_in_kernel) == (256, 128, 2, 1), (m, n, k)


def test_one_k_block_takes_a_small_tile(pkg):
    """K = 128 is all first copies and output: 64x64 where the chip holds those tiles at once, else 128x128 in four waves."""
    for m, n, tile in [(1, 115, 64), (2944, 171, 64), (640, 575, 64), (107, 6464, 64), (13653, 64, 64), (8576, 2624, 128), (10880, 1484, 128), (9106, 256, 128), (8192, 8192, 128)]:
        p = pkg.plan(m, n, 128)
        assert (p.tile_m, p.tile_n, p.split_k, p.block_threads) == (tile, tile, 1, 256), (m, n)


def test_small_products_take_one_launch_where_that_is_faster(pkg):
    """A second launch costs a caller 2.5 to 4 us: with 12 to 15 K blocks more than the K split behind it saves."""
    for m, n, k in [(12, 128, 1536), (12, 512, 1536), (8, 576, 1664), (64, 512, 1536), (4, 832, 1792), (21, 576, 1792), (200, 128, 1536)]:
        p = pkg.plan(m, n, k)
        assert p.split_k == 1 or p.sum_in_kernel, (m, n, k)
    for m, n, k in [(1, 512, 7168), (12, 512, 5632), (64, 512, 7168)]:
        p = pkg.plan(m, n, k)
        assert p.split_k >= 4 and not p.sum_in_kernel, (m, n, k)


@pytest.mark.parametrize("m,n,k", [(64, 512, 1536), (64, 512, 2048), (1, 1088, 1664), (32, 512, 2048), (64, 2304, 2048), (256, 512, 1024)])
def test_a_plan_of_the_waves_tiles_says_what_runs(pkg, m, n, k):
    """One launch and no workspace at every number of K blocks: nothing for a caller to allocate, and nothing that is refused without."""
    p = pkg.plan(m, n, k)
    assert p.variant == 12 and p.form >= 2
    assert (p.sum_in_kernel, p.workspace_bytes, pkg.workspace_bytes(m, n, k)) == (int(p.split_k > 1), 0, 0)
    assert p.split_k == (8 if k > 1024 else 1)


def test_waves_tiles_in_one_round_only(pkg):
    """The tiles that hold all K partitions are planned where all their workgroups are on the chip at once (256 of 32x64, 512 of 16x64):
    sizes measured 4 to 36 % slower in two rounds, and sizes at the edge that are faster."""
    for m, n, k in [(320, 1664, 384), (612, 896, 256), (64, 8448, 256), (20, 17920, 896), (2130, 242, 256), (4203, 126, 256), (28, 17878, 384), (867, 637, 256)]:
        p = pkg.plan(m, n, k)
        assert not (p.variant == 12 and p.form >= 2), (m, n, k)
    for m, n, k in [(8000, 64, 256), (256, 512, 1024), (18, 13764, 896), (41, 8128, 256)]:
        p = pkg.plan(m, n, k)
        assert p.variant == 12 and p.form >= 2 and p.grid_x <= 163840 // p.lds_bytes * 256, (m, n, k)


@pytest.mark.parametrize("m,n,k,tile,split", [(1024, 512, 7168, (64, 128), 4), (86, 3392, 5632, (64, 128), 4), (107, 3520, 4736, (64, 64), 2), (384, 1728, 3840, (64, 64), 1),
                                              (92, 3478, 4480, (64, 64), 2), (1115, 1088, 2944, (64, 128), 1), (619, 768, 6272, (64, 64), 2), (565, 640, 6656, (64, 128), 4),
                                              (112, 3712, 6144, (64, 128), 4), (891, 768, 4864, (64, 128), 3), (250, 4096, 7168, (128, 128), 4), (1024, 1536, 7168, (128, 128), 2)])
def test_many_partitions_of_full_tiles_are_not_planned_for_a_shared_sum(pkg, m, n, k, tile, split):
    """Six and eight partitions of full 128x128 tiles, three of few K blocks: 4 to 40 % slower, operands from HBM and from the caches, than
    the plans here; and two sizes where sharing the sum pays."""
    p = pkg.plan(m, n, k)
    assert ((p.tile_m, p.tile_n), p.split_k) == (tile, split)


def test_an_incomplete_binding_is_named(pkg, monkeypatch):
    """A CPython binding built before a function was added to it gives way to ctypes with a warning that says so."""
    lib_mod, whole = pkg._lib, pkg._lib.pycall()
    stale = types.SimpleNamespace(**{name: getattr(whole, name) for name in lib_mod._CALLS if name not in ("quantize_a", "moe_route")})
    monkeypatch.setattr(lib_mod, "_pycall", stale)
    monkeypatch.setattr(lib_mod, "_calls", None)
    with pytest.warns(UserWarning, match="quantize_a, moe_route"):
        calls = lib_mod.calls()
    assert all(hasattr(calls, name) for name in lib_mod._CALLS)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert lib_mod.calls() is calls                                     # once
