"""The layer call's host side in C++ loads beside torch without slowing it down."""
import importlib.util
import os
import struct
import subprocess

import pytest

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
