"""Where the arrays of LDS start that kernels fill 16 bytes at a time: dynamic LDS follows a kernel's static LDS, whose size the compiler
rounds up to the alignment that the dynamic array is declared with and writes into the code object.  And how much of it a kernel may ask for."""
import glob
import os
import re
import struct

import pytest

from drone_amd import _lib

BUNDLE, NOTE = b"__CLANG_OFFLOAD_BUNDLE__", b"AMDGPU\0"


def _kernels():
    """Metadata of the library's kernels: the msgpack notes of its gfx950 code objects."""
    msgpack = pytest.importorskip("msgpack")
    blob = open(_lib.library_path(), "rb").read()
    at = blob.find(BUNDLE)
    while at >= 0:
        entry = at + len(BUNDLE) + 8
        for _ in range(struct.unpack_from("<Q", blob, entry - 8)[0]):
            offset, size, name_size = struct.unpack_from("<QQQ", blob, entry)
            name = blob[entry + 24:entry + 24 + name_size]
            entry += 24 + name_size
            code = blob[at + offset:at + offset + size] if b"gfx950" in name else b""
            note = code.find(NOTE)
            while note >= 0:
                name_bytes, bytes_, kind = struct.unpack_from("<III", code, note - 12)
                if name_bytes == len(NOTE) and kind == 32:  # NT_AMDGPU_METADATA
                    yield from msgpack.unpackb(code[note + 8:note + 8 + bytes_], strict_map_key=False)["amdhsa.kernels"]
                    break
                note = code.find(NOTE, note + 1)
        at = blob.find(BUNDLE, at + 1)


def test_hot_sources_start_at_16_bytes():
    sizes = {k[".name"]: k[".group_segment_fixed_size"] for k in _kernels()}
    hot = {name: size for name, size in sizes.items() if "sell_iterate_hot_kernel" in name or "sell_push_kernel" in name}
    assert len(hot) == 2
    assert all(size % 16 == 0 for size in hot.values()), hot
    assert all(size + 160_000 <= 163_840 for size in hot.values()), hot


def test_limits_of_dynamic_lds_are_constants():
    """The limit that hipFuncSetAttribute sets belongs to the kernel, not to the handle that sets it: were it a handle's own size, a handle
    made later with a smaller one would leave too low a limit behind for those made before."""
    limits = []
    for path in glob.glob(os.path.join(os.path.dirname(_lib.library_path()), "*.hip")):
        limits += re.findall(r"hipFuncAttributeMaxDynamicSharedMemorySize,\s*(?:\(int\))?([^()\s]+)\)", open(path).read())
    assert len(limits) >= 6
    assert all(re.fullmatch(r"k[A-Z]\w*", limit) for limit in limits), limits
