"""Compiles and runs the host check of the wait counts with four buffers of C per wave (plain g++, no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_group_of_c_in_one_of_four_buffers_has_landed_when_it_is_read(tmp_path):
    exe = tmp_path / "copy_waits_buffers_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), os.path.join(ROOT, "tests", "host", "copy_waits_buffers_check.cpp")])
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0 and "copy waits OK" in res.stdout, res.stdout
