"""The layer call's host side in C++ loads beside torch without slowing it down."""
import struct

import triton_int8_amd as T

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
