"""Plans and forced arguments that name one of the two forms of a variant, or a K split: honoured or refused, never
something else run in their place.  Host checks only: every call here returns before a launch."""
import ctypes

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
