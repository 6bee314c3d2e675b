"""Compiles and runs the host check of how a batch is cut into launches (plain g++, no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_batches_of_any_size_are_cut_into_launches(tmp_path):
    exe = tmp_path / "launch_limits_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-o", str(exe), os.path.join(ROOT, "tests", "host", "launch_limits_check.cpp")])
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0 and "launch limits OK" in res.stdout, res.stdout


def test_sample_kernels_launch_through_it():
    source = open(os.path.join(ROOT, "rocwmma_amd", "csrc", "dlrm_sample.hip")).read()
    assert source.count("hipLaunchKernelGGL") == 2 and source.count("forEachLaunch(") == 2
