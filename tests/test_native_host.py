"""The native autograd library: what serves where it is missing, broken or stale."""

import pytest

from neuronx_distributed_amd import ops
from neuronx_distributed_amd.ops import build


@pytest.fixture
def native(monkeypatch):
    """``ops._native_flash`` as a process finds it that has not asked yet."""
    monkeypatch.setattr(ops, "_require_lib", lambda: None)
    return ops._native_flash.__wrapped__


def test_a_library_that_does_not_load_leaves_calls_to_python(monkeypatch, tmp_path,
                                                             native):
    lib = tmp_path / "libnxd_host.so"
    monkeypatch.setattr(build, "HOST_LIB", str(lib))
    assert native() is None                        # not there: no word about it
    lib.write_bytes(b"of another machine")
    with pytest.warns(UserWarning, match="does not load"):
        assert native() is None
