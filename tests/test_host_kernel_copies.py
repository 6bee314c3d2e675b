"""Copies into LDS of the built kernels: one instruction each.  Where the compiler has a copy's descriptor or offset in vector registers, though all
lanes have the same, it makes a loop over the lanes' values of it."""
import os
import subprocess

import pytest

import rocwmma_amd.api as api
from test_host_kernel_resources import device_objects

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def looped_copies(lines):
    """Kernels with a copy (buffer_load ... lds) between an s_and_saveexec and a branch back for the lanes that are left."""
    found, kernel, masked, copied = {}, None, False, False
    for line in lines:
        if line.endswith(">:\n"):
            kernel, masked, copied = line.split("<")[1][:-3], False, False
        elif "s_and_saveexec_b64" in line:
            masked, copied = True, False
        elif "buffer_load" in line and " lds" in line:
            copied = masked
        elif "s_cbranch" in line or "s_branch" in line:
            if copied and "s_cbranch_execnz" in line:
                found[kernel] = found.get(kernel, 0) + 1
            masked = copied = False
    return found


def test_the_pattern():
    loop = ["0 <kernel>:\n", "v_readfirstlane_b32 s24, v65\n", "s_and_saveexec_b64 s[10:11], s[10:11]\n",
            "buffer_load_dwordx4 v64, s[16:19], s24 offen lds\n", "s_xor_b64 exec, exec, s[10:11]\n", "s_cbranch_execnz 65533\n"]
    assert looped_copies(loop) == {"kernel": 1}
    assert looped_copies(loop[:1] + loop[3:]) == {} and looped_copies(loop[:3] + loop[4:]) == {}


def test_no_copy_is_a_loop_over_lanes(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("needs llvm-objdump of the ROCm toolchain")
    kernels, looped = 0, {}
    for i, obj in enumerate(device_objects(api.library_path())):
        elf = tmp_path / f"{i}.elf"
        elf.write_bytes(obj)
        dump = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", str(elf)], stdout=subprocess.PIPE, text=True)
        looped.update(looped_copies(dump.stdout))
        assert dump.wait() == 0
        kernels += 1
    assert kernels > 0
    assert not looped, looped
