"""Registers of the table update as it is launched by default (512 threads):
none are spilled to memory, in any of its forms (read from the metadata of the
library's own code objects)."""
import struct

import pytest

from glint_pipeline_amd import runtime

msgpack = pytest.importorskip("msgpack")


def kernels():
    """{mangled name: metadata} of the kernels in the built library."""
    data = runtime.LIB_PATH.read_bytes()
    found, at = {}, data.find(b"\x7fELF", 4)
    while at >= 0:
        if data[at + 18:at + 20] == struct.pack("<H", 224):   # an AMD GPU's code
            phoff, = struct.unpack_from("<Q", data, at + 32)
            size, count = struct.unpack_from("<HH", data, at + 54)
            for k in range(count):
                kind, = struct.unpack_from("<I", data, at + phoff + k * size)
                off, = struct.unpack_from("<Q", data, at + phoff + k * size + 8)
                if kind != 4:   # notes
                    continue
                nlen, dlen, note = struct.unpack_from("<III", data, at + off)
                name = data[at + off + 12:at + off + 12 + nlen].rstrip(b"\0")
                desc = at + off + 12 + (nlen + 3) // 4 * 4
                if name == b"AMDGPU" and note == 32:
                    for m in msgpack.unpackb(data[desc:desc + dlen])["amdhsa.kernels"]:
                        found[m[".name"]] = m
        at = data.find(b"\x7fELF", at + 4)
    return found


def test_table_update_spills_nothing():
    if not runtime.LIB_PATH.exists():
        pytest.skip("the library is not built")
    table = {n: m for n, m in kernels().items() if "k_tableILb" in n or "kf_tableILb" in n}
    default = {n: m for n, m in table.items() if "ELi512E" in n}
    assert len(table) == 12 and len(default) == 4
    for name, m in default.items():
        assert m[".vgpr_spill_count"] == 0 and m[".private_segment_fixed_size"] == 0, name
