"""Registers of the built kernels, from the metadata the compiler leaves in the library: they may not spill.  (The stream-K
kernels hold the accumulators of a 256 x 256 tile through their hand-over and spill around it.)"""
import os
import struct
import subprocess

import pytest

import rocwmma_amd.api as api

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
STREAMK_SPILLS = 256


def device_objects(path):
    """The gfx950 code objects of every translation unit's offload bundle."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(MAGIC, at + len(MAGIC))


def test_no_kernel_spills_registers(tmp_path):
    if not os.path.exists(READELF):
        pytest.skip("needs llvm-readelf of the ROCm toolchain")
    kernels, spilled = 0, []
    for i, obj in enumerate(device_objects(api.library_path())):
        elf = tmp_path / f"{i}.elf"
        elf.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(elf)], stdout=subprocess.PIPE, text=True, check=True).stdout
        name = None
        for line in notes.splitlines():
            key, _, value = line.strip().partition(":")
            if key == ".name" and not value.strip().startswith("__"):
                name = value.strip()
            if key == ".vgpr_spill_count":
                kernels += 1
                if int(value) > (STREAMK_SPILLS if "gemmStreamKKernel" in name else 0):
                    spilled.append((name, int(value)))
    assert kernels > 0
    assert not spilled, spilled
