"""What the built library's kernels use, from the metadata that the compiler left in it (no GPU)."""
import os
import struct

import pytest

import fastlanes_amd as fa

msgpack = pytest.importorskip("msgpack")


def _kernels(path):
    """Metadata of every kernel in a library's code objects."""
    with open(path, "rb") as f:
        d = f.read()
    out, i = [], d.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while i >= 0:
        at = i + 32
        for _ in range(struct.unpack_from("<Q", d, i + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", d, at)
            target, at = d[at + 24: at + 24 + n], at + 24 + n
            if b"gfx950" not in target or not size:
                continue
            elf = d[i + off: i + off + size]
            table, = struct.unpack_from("<Q", elf, 40)
            esize, count = struct.unpack_from("<HH", elf, 58)
            for k in range(count):
                kind, = struct.unpack_from("<I", elf, table + k * esize + 4)
                if kind != 7:  # SHT_NOTE
                    continue
                note, = struct.unpack_from("<Q", elf, table + k * esize + 24)
                name, desc, _ = struct.unpack_from("<III", elf, note)
                out += msgpack.unpackb(elf[note + 12 + (name + 3) // 4 * 4:][:desc])["amdhsa.kernels"]
        i = d.find(b"__CLANG_OFFLOAD_BUNDLE__", i + 1)
    return out


@pytest.mark.skipif(not os.path.exists(fa.LIB_PATH), reason="library not built")
def test_string_kernels_do_not_spill():
    """No string kernel has scratch or spilled registers: builds that spilled decoded some segments wrong."""
    seen = [k for k in _kernels(fa.LIB_PATH) if "k_fsst" in k[".name"]]
    assert len(seen) == 6  # the scan, two forms of the count, three of the decode
    for k in seen:
        used = {f: k[f] for f in (".private_segment_fixed_size", ".vgpr_spill_count", ".sgpr_spill_count")}
        assert not any(used.values()), (k[".name"], used)
