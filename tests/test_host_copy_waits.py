"""Compiles and runs the host check of the wait counts for copies into LDS (plain g++, no GPU)."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_staged_group_of_c_has_landed_when_it_is_read(tmp_path):
    exe = tmp_path / "copy_waits_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), os.path.join(ROOT, "tests", "host", "copy_waits_check.cpp")])
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0 and "copy waits OK" in res.stdout, res.stdout


def test_no_wait_for_copies_counts_stores():
    """Stores of D are no copies: no wait of the blocked GEMM may leave any of them in its count."""
    source = open(os.path.join(ROOT, "rocwmma_amd", "csrc", "gemm_blocked_core.hpp")).read()
    waits = re.findall(r"waitCopiesAndReads<(.*?)>\(\)", source)
    assert waits and not [w for w in waits if "Stores" in w], waits
