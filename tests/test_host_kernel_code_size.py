"""Code of the built kernels that a call on operands not used before waits for: the fused epilogue of a 256 x 256 tile on four waves does not
write the activation out for every result of a lane (256 of them: 86 to 131 KB, with one wave per SIMD and nobody to cover the fetches)."""
import os
import subprocess

import pytest

import rocwmma_amd.api as api
from test_host_kernel_resources import READELF, device_objects

INSTRUCTION_CACHE = 65536  # bytes, shared by two compute units


def test_fused_kernels_on_wide_waves_fit_the_instruction_cache(tmp_path):
    if not os.path.exists(READELF):
        pytest.skip("needs llvm-readelf of the ROCm toolchain")
    kernels, large = 0, []
    for i, obj in enumerate(device_objects(api.library_path())):
        elf = tmp_path / f"{i}.elf"
        elf.write_bytes(obj)
        for line in subprocess.run([READELF, "-s", "-W", str(elf)], stdout=subprocess.PIPE, text=True, check=True).stdout.splitlines():
            field = line.split()
            # (Waves M, N 2 x 2, blocks 8 x 8, fused; the kernel of whole rounds: one tile's code)
            if len(field) == 8 and field[3] == "FUNC" and "gemmBlockedKernel" in field[7] and "Lj2ELj2ELj8ELj8ELj2ELj1ELj16ELb0ELb0ELb1E" in field[7]:
                kernels += 1
                if int(field[2]) > INSTRUCTION_CACHE:
                    large.append((field[7], int(field[2])))
    assert kernels > 0
    assert not large, large
