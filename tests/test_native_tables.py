"""The tables of sizes that the native calls may take."""
import importlib


def test_sizes_of_many_batches_are_kept(monkeypatch):
    """A layer has two products: 1000 batch sizes are 2000 sizes, and all of them stay with the native call.  The table is bounded."""
    sub = importlib.import_module("amd-developer-challenge-2025_amd.submission")
    monkeypatch.setattr(sub, "_checked_experts", {})
    sizes = [(silu, 8, rows, 512, 256) for rows in range(1, 1001) for silu in (True, False)]
    for size in sizes:
        sub._remember(*size, 0)
    assert all((int(silu), *rest) in sub._checked_experts for silu, *rest in sizes)
    for rows in range(1, 20000):
        sub._remember(False, 16, rows, 512, 256, 0)
    assert len(sub._checked_experts) <= sub._CHECKED_MAX <= 8192
