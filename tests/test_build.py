"""What make builds without torch, when it rebuilds the native bindings, and what the loader says
to a library of another ABI version or bindings of another torch (CPU)."""
import os
import shutil
import subprocess
import warnings

import pytest
import torch

from needle_amd import _lib

CSRC = _lib.LIB_PATH.parent / "csrc"


def _plan(*args):
    """The commands make would run (none of them is)."""
    return subprocess.run(["make", "-n", "-C", str(CSRC), *args], text=True, check=True,
                          capture_output=True).stdout


def test_the_library_alone_without_torch(tmp_path):
    python = tmp_path / "python"   # an interpreter that has no torch
    python.write_text("#!/bin/sh\nexit 1\n")
    python.chmod(0o755)
    out = _plan(f"PYTHON={python}", f"OUT={tmp_path}/lib.so", f"NATIVE={tmp_path}/n.so")
    assert "bind.cpp" not in out and "lib.so" in out and "not built" in out
    assert "bind.cpp" in _plan(f"NATIVE={tmp_path}/n.so")


def test_another_torch_rebuilds_the_bindings(tmp_path):
    native = tmp_path / "n.so"
    native.touch()
    os.utime(native, (4e9, 4e9))       # newer than every source
    args = (f"NATIVE={native}", "TORCH_VERSION=0.0.0+other")
    assert "bind.cpp" in _plan(*args) and "native-0.0.0+other" in _plan(*args)


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not installed")
def test_an_older_library_is_refused_by_its_version(tmp_path, monkeypatch):
    src = tmp_path / "old.c"
    src.write_text("int ndl_abi_version(void) { return 8; }\n")
    lib = tmp_path / "libold.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    monkeypatch.setenv("NEEDLE_AMD_LIB", str(lib))
    monkeypatch.setattr(_lib, "_LIB", None)
    with pytest.raises(_lib.NeedleAmdError, match="ABI version 8"):
        _lib.load()


def test_bindings_of_another_torch_are_left_alone(monkeypatch):
    lib = _lib.load()
    native = pytest.importorskip("needle_amd._native")
    assert native.torch_version == torch.__version__
    monkeypatch.setattr(native, "torch_version", "0.0.0+other")
    monkeypatch.setattr(_lib, "NATIVE", None)
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        _lib._load_native(lib)
    assert _lib.NATIVE is None and any("0.0.0+other" in str(w.message) for w in seen)
