"""The native autograd library: what serves where it is missing, broken or stale."""

import os
import re
import shutil

import pytest
import torch

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
    monkeypatch.setattr(build, "host_lib", lambda: str(lib))
    monkeypatch.setattr(build, "host_libs", lambda: [])
    assert native() is None                        # not there: no word about it
    lib.write_bytes(b"of another machine")
    with pytest.warns(UserWarning, match="does not load"):
        assert native() is None


def test_a_library_of_other_sources_or_another_torch_is_not_loaded(
        monkeypatch, tmp_path, native):
    """A new torch, another source and other prototypes each ask for a library of their
    own; one that is left of before is not loaded and not taken as built."""
    csrc = tmp_path / "csrc"
    shutil.copytree(build.CSRC, csrc)
    monkeypatch.setattr(build, "CSRC", str(csrc))
    monkeypatch.setattr(build, "_THIS", str(tmp_path))
    names = {build.host_lib()}
    monkeypatch.setattr(torch, "__version__", "1.0")
    names.add(build.host_lib())
    for path in (csrc / "host" / "flash_autograd.cpp", csrc / "flash_attn.h"):
        path.write_text(path.read_text() + "\n")
        names.add(build.host_lib())
    assert len(names) == 4
    (tmp_path / "libnxd_host.so").write_bytes(b"of before")
    asked = []
    monkeypatch.setattr(torch.ops, "load_library", asked.append)
    with pytest.warns(UserWarning, match="another torch"):
        assert native() is None
    assert not asked

    def compile_to(cmd, verbose):
        open(cmd[cmd.index("-o") + 1], "wb").close()

    monkeypatch.setattr(build, "_run", compile_to)
    assert build.host_libs() != [build.host_lib()]
    build.build_host(verbose=False)
    assert build.host_libs() == [build.host_lib()]


def test_a_build_without_a_host_compiler_ends_well(monkeypatch, tmp_path, capsys):
    """Kernels are what a build has to make; Python's functions serve beside them."""
    monkeypatch.setattr(build, "build_group", lambda *a: None)
    monkeypatch.setattr(build, "_THIS", str(tmp_path))
    monkeypatch.setenv("PATH", str(tmp_path))          # no g++
    assert build.build(force=True, verbose=False) == build.LIB
    assert "Python's functions serve" in capsys.readouterr().err
    assert not build.host_libs()
    gxx = tmp_path / "g++"                             # one without torch's headers
    gxx.write_text("#!/bin/sh\nexit 1\n")
    gxx.chmod(0o755)
    build.build(force=True, verbose=False)
    assert "g++ failed (1)" in capsys.readouterr().err


def test_prototypes_are_in_one_place():
    """Callers and kernels include them, so a signature cannot change on one side."""
    for name in ("host/flash_autograd.cpp", "flash_attn.hip", "flash_attn_bwd.hip"):
        with open(os.path.join(build.CSRC, name)) as f:
            text = f.read()
        assert re.search(r'#include "(\.\./)?flash_attn\.h"', text), name
        if name.endswith(".cpp"):
            assert 'extern "C"' not in text
