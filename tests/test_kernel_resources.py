"""What the compiler gave the kernels of the built library (no GPU)."""
import os
import re
import struct

import pytest

from ed_lattice_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _library():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    with open(_lib.LIB_PATH, "rb") as f:
        return f.read()


def _device_code(d):
    """(start, size) of the gfx950 code object in the offload bundle."""
    at = d.index(b"__CLANG_OFFLOAD_BUNDLE__")
    (n,) = struct.unpack_from("<Q", d, at + 24)
    pos = at + 32
    for _ in range(n):
        off, size, ln = struct.unpack_from("<QQQ", d, pos)
        if b"gfx950" in d[pos + 24:pos + 24 + ln]:
            return at + off, size
        pos += 24 + ln
    raise AssertionError("no gfx950 code in the library")


def _kernels(d):
    """The kernels' metadata from the code object's notes."""
    at, size = _device_code(d)
    e = d[at:at + size]
    (shoff,) = struct.unpack_from("<Q", e, 40)
    entsize, num = struct.unpack_from("<HH", e, 58)
    for k in range(num):
        _, kind, _, _, off, n = struct.unpack_from("<IIQQQQ", e, shoff + k * entsize)
        if kind != 7:  # SHT_NOTE
            continue
        namesz, descsz, ntype = struct.unpack_from("<III", e, off)
        if ntype == 32:  # NT_AMDGPU_METADATA
            start = off + 12 + (namesz + 3) // 4 * 4
            return msgpack.unpackb(e[start:start + descsz])["amdhsa.kernels"]
    raise AssertionError("no kernel metadata")


def test_up_pass_without_scratch():
    """The up pass keeps its values in registers: the operator's launches and both
    forms of a chain's.  (Not three fp64 columns of two rows and eight hops, more
    than the 128 registers a thread of 1024 has, which a tuner times like the rest.)"""
    ks = [k for k in _kernels(_library()) if "k_pass_up" in k[".name"] and "IdLi3ELi2ELi8E" not in k[".name"]]
    assert len(ks) > 100
    bad = {k[".name"]: k[".private_segment_fixed_size"] for k in ks if k[".private_segment_fixed_size"]}
    assert not bad, bad


def test_host_and_device_code_match():
    """Every kernel the host side launches is in the device code: the library was
    built from one state of the sources."""
    d = _library()
    at, size = _device_code(d)
    device = {k[".name"].encode() for k in _kernels(d)}
    host = set(re.findall(rb"\x00(_ZN3edl\d+k_\w+)\x00", d[:at] + d[at + size:]))
    assert len(host) > 100 and host <= device, sorted(host - device)[:5]
