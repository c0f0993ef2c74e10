"""Registers of the built kernels, from the code objects' own metadata."""
import os
import struct
import subprocess

import pytest

from epure.kernels import _abi

msgpack = pytest.importorskip("msgpack")


def kernels(path):
    """{demangled name: metadata} of every gfx950 kernel in a HIP library:
    the amdhsa note (type 32) of the ELF code objects in its offload bundles."""
    data = open(path, "rb").read()
    found, pos = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while pos >= 0:
        count, at = struct.unpack_from("<Q", data, pos + 24)[0], pos + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in target and size:
                found.update(_notes(data[pos + offset:pos + offset + size]))
        pos = data.find(b"__CLANG_OFFLOAD_BUNDLE__", pos + 1)
    names = subprocess.run(["c++filt"], input="\n".join(found), text=True, capture_output=True, check=True)
    return dict(zip(names.stdout.splitlines(), found.values()))


def _notes(elf):
    table, (entry, count) = struct.unpack_from("<Q", elf, 0x28)[0], struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        head = table + i * entry
        if struct.unpack_from("<I", elf, head + 4)[0] != 7:     # SHT_NOTE
            continue
        at, size = struct.unpack_from("<QQ", elf, head + 24)
        end = at + size
        while at < end:
            name, desc, kind = struct.unpack_from("<III", elf, at)
            body = at + 12 + (name + 3) // 4 * 4
            if kind == 32:
                meta = msgpack.unpackb(elf[body:body + desc], strict_map_key=False)
                for k in meta["amdhsa.kernels"]:
                    yield k[".name"], k
            at = body + (desc + 3) // 4 * 4


def test_64_row_prefill_tiles_fit_two_workgroups_per_cu():
    """The 64-row tile on eight waves is planned as two workgroups per CU
    (K is split towards twice the CUs): four waves on each of a SIMD's 512
    registers a lane, 128 each, nothing spilled, and half of 160 KiB of LDS."""
    meta = kernels(_abi.LIB_PATH)
    tiles = {n: k for n, k in meta.items() if "pf_kernel<" in n and ", 64, 4, 1, 8, " in n}
    assert len(tiles) == 2 * 2 * 2 * 2          # bits, grouped, f32 scales, groups of 128
    for name, k in tiles.items():
        assert k[".vgpr_count"] <= 128, name
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name
        assert k[".group_segment_fixed_size"] <= 80 * 1024, name
