"""The library's version moves with what it accepts.  Host check only."""


def test_the_grouped_tile_has_a_version(pkg):
    """A caller that forces the 128x256 tile of grouped calls can tell a library that takes it (401) from one that refuses it (400)."""
    assert pkg._lib.load().fp8bs_version() >= 401
