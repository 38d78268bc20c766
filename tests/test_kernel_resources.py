"""No kernel of the built library keeps vector registers in scratch
memory: such a spill shows in no result, only in time. Read from the metadata
note that the compiler leaves in this repository's own code object."""

from __future__ import annotations

import struct

import msgpack

from ternel_amd.build import ARCH, LIB_PATH

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def code_object() -> bytes:
    data = LIB_PATH.read_bytes()
    start = data.index(BUNDLE)
    (count,) = struct.unpack_from("<Q", data, start + len(BUNDLE))
    at = start + len(BUNDLE) + 8
    for _ in range(count):
        offset, size, length = struct.unpack_from("<QQQ", data, at)
        name = data[at + 24:at + 24 + length].decode()
        at += 24 + length
        if name.endswith(ARCH):
            return data[start + offset:start + offset + size]
    raise AssertionError(f"no {ARCH} code object in {LIB_PATH}")


def kernels(elf: bytes) -> list[dict]:
    (sections,) = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        _, kind, _, _, offset, size = struct.unpack_from("<IIQQQQ", elf, sections + i * entry)
        if kind != 7:  # SHT_NOTE
            continue
        at = offset
        while at < offset + size:
            name, desc, note = struct.unpack_from("<III", elf, at)
            at += 12 + (name + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                return msgpack.unpackb(elf[at:at + desc], raw=False)["amdhsa.kernels"]
            at += (desc + 3) // 4 * 4
    raise AssertionError("no metadata note")


def test_no_kernel_spills_vector_registers() -> None:
    found = kernels(code_object())
    names = [k[".name"] for k in found]
    for stem in ("trit_gemm_kernel", "wide_gemm_kernel", "lut_gemv_kernel", "mfma_gemm_kernel"):
        assert any(stem in name for name in names), stem
    spilled = {k[".name"]: k[".vgpr_spill_count"] for k in found if k[".vgpr_spill_count"]}
    assert not spilled, spilled
