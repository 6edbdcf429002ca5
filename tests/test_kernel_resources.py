"""What the compiler reports about the kernels of the built library (the notes of its code objects)."""
import importlib.util
import os
import struct

import msgpack

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _kernels():
    spec = importlib.util.spec_from_file_location("build_of_the_library", os.path.join(ROOT, "project-currennt-public_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    with open(build.LIB_PATH, "rb") as f:
        data = f.read()
    found, at = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        pos = at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if target.startswith(b"hip") and size:
                found.update(_notes(data[at + offset:at + offset + size]))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return found


def _notes(elf):
    table, = struct.unpack_from("<Q", elf, 0x20)
    entry, count = struct.unpack_from("<HH", elf, 0x36)
    for i in range(count):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, table + i * entry)
        pos = offset
        while kind == 4 and pos < offset + size:  # PT_NOTE
            name, desc, note = struct.unpack_from("<III", elf, pos)
            body = pos + 12 + (name + 3) // 4 * 4
            if note == 32:  # AMDGPU metadata
                for k in msgpack.unpackb(elf[body:body + desc], strict_map_key=False)["amdhsa.kernels"]:
                    yield k[".name"], k
            pos = body + (desc + 3) // 4 * 4


def test_no_product_kernel_spills_registers():
    kernels = {n: k for n, k in _kernels().items() if "gemm_split_kernel" in n}
    assert len(kernels) >= 40
    spilled = {n: k[".vgpr_spill_count"] for n, k in kernels.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not spilled
