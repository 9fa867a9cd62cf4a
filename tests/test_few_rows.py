"""Products of a few rows: which of them the weight-streaming kernels take."""

import types

from neuronx_distributed_amd.ops import serving as sv


def test_a_library_without_the_products_is_not_used(monkeypatch):
    """One that was built before they came is there, but has none."""
    monkeypatch.setattr(sv, "_LIB", types.SimpleNamespace())
    assert not sv.available()
    monkeypatch.setattr(sv, "_LIB",
                        types.SimpleNamespace(sv_stream_linear=None))
    assert sv.available()
