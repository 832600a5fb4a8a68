"""The layer call's host side in C++ loads beside torch without slowing it down."""
import ctypes
import importlib.util
import os
import struct
import subprocess
import sys

import pytest
import torch

import triton_int8_amd as T
from conftest import ROOT

PT_TLS = 7


def test_no_thread_local_storage():
    """A loaded library whose thread-local variables nobody touches makes every other access to such variables slow (glibc)."""
    data = open(T._lib.NATIVE_PATH, "rb").read()
    assert data[:5] == b"\x7fELF\x02"
    offset, = struct.unpack_from("<Q", data, 32)
    size, count = struct.unpack_from("<HH", data, 54)
    kinds = [struct.unpack_from("<I", data, offset + i * size)[0] for i in range(count)]
    assert 1 in kinds and PT_TLS not in kinds


def test_loaded_on_this_torch():
    assert T._lib.native() is not None


@pytest.mark.parametrize("other", ["torch", "python", "arguments", "problems"])
def test_built_for_something_else(monkeypatch, other):
    """Another torch or Python may resolve all its symbols and still keep its fields elsewhere."""
    monkeypatch.setattr(T._lib, "_native", None)
    longer = lambda base: type(base.__name__, (ctypes.Structure,), {"_fields_": [*base._fields_, ("more", ctypes.c_int64)]})
    with monkeypatch.context() as m:
        if other == "torch":
            m.setattr(torch, "__version__", torch.__version__ + ".1")
        elif other == "python":
            m.setattr(sys, "version_info", (sys.version_info[0], sys.version_info[1] + 1, 0))
        else:
            name = "LinearArgs" if other == "arguments" else "GemmProblem"
            m.setattr(T._lib, name, longer(getattr(T._lib, name)))
        assert T._lib.native() is None
    T._lib._native = None
    assert T._lib.native() is not None


@pytest.mark.parametrize("failure", ["no compiler", "no headers"])
def test_library_is_built_without_it(monkeypatch, tmp_path, capsys, failure):
    """A machine with hipcc alone gets the library, and no extension of an earlier build is left beside it."""
    spec = importlib.util.spec_from_file_location("ti8_build", os.path.join(ROOT, "triton-int8_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    monkeypatch.setattr(build, "LIB", str(tmp_path / "libti8.so"))
    monkeypatch.setattr(build, "NATIVE", str(tmp_path / "_native.so"))
    (tmp_path / "_native.so").write_bytes(b"")

    def run(cmd, **_):
        if cmd[0] != "g++":
            return subprocess.CompletedProcess(cmd, 0, "")
        if failure == "no compiler":
            raise FileNotFoundError("g++")
        return subprocess.CompletedProcess(cmd, 1, "fatal error: torch/csrc/Exceptions.h: No such file or directory")
    monkeypatch.setattr(build.subprocess, "run", run)
    assert build.build() == build.LIB
    assert not os.path.exists(build.NATIVE) and "not built" in capsys.readouterr().err
