"""What the compiler says of the built kernels: none of them spills vector registers or uses scratch memory."""
import struct

import pytest

from flexgemm_amd import build

msgpack = pytest.importorskip("msgpack")


def _kernels(path):
    """{mangled name: metadata} of every gfx950 kernel in a shared library (ELF images inside its fat binary, AMDGPU metadata notes)."""
    raw, found, at = open(path, "rb").read(), {}, 0
    while (at := raw.find(b"\x7fELF\x02\x01", at + 1)) > 0:
        if struct.unpack_from("<H", raw, at + 18)[0] != 224:           # EM_AMDGPU
            continue
        table, = struct.unpack_from("<Q", raw, at + 40)
        size, count = struct.unpack_from("<HH", raw, at + 58)
        for i in range(count):
            kind, offset, length = (struct.unpack_from(f, raw, at + table + i * size + o)[0] for f, o in (("<I", 4), ("<Q", 24), ("<Q", 32)))
            pos, end = at + offset, at + offset + length
            while kind == 7 and pos + 12 <= end:                       # SHT_NOTE
                name, desc, note = struct.unpack_from("<III", raw, pos)
                body = pos + 12 + (name + 3) // 4 * 4
                if note == 32:                                         # NT_AMDGPU_METADATA
                    for k in msgpack.unpackb(raw[body:body + desc])["amdhsa.kernels"]:
                        found[k[".name"]] = k
                pos = body + (desc + 3) // 4 * 4
    return found


def test_no_register_is_spilled():
    mine = {k: v for k, v in _kernels(build.build(verbose=False)).items() if k.startswith("_ZN3fgx")}
    assert any("stem_wgrad_kernel" in k for k in mine)
    assert {k: v[".vgpr_spill_count"] for k, v in mine.items() if v[".vgpr_spill_count"] or v[".private_segment_fixed_size"]} == {}
