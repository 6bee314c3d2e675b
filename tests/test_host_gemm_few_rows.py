"""Which problems the kernel whose waves share K takes, and on which tile (plain g++, no GPU)."""
import os
import subprocess

from few_rows import CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def few_of(tmp_path, problems):
    exe = tmp_path / "few_of"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), os.path.join(ROOT, "tests", "host", "few_of.cpp")])
    asked = "".join("%d %d %d %d %d\n" % p for p in problems)
    out = subprocess.run([str(exe)], input=asked, stdout=subprocess.PIPE, text=True, check=True).stdout
    return [tuple(int(x) for x in line.split()) for line in out.splitlines()]


def test_cases_run_on_the_tiles_they_name(tmp_path):
    got = few_of(tmp_path, [(kind, m, n, k, out) for kind, _, _, m, n, k, out in CASES])
    wrong = [(case, tile) for case, tile in zip(CASES, got) if case[1:3] != tile]
    assert not wrong, wrong


def test_wide_weights_and_short_k_stay_with_the_blocked_kernel(tmp_path):
    assert few_of(tmp_path, [(0, 128, 14336, 8192, 2), (0, 64, 14336, 8192, 4), (1, 128, 14336, 4096, 4), (2, 96, 8192, 1024, 4), (0, 16, 256, 64, 4)]) == [(0, 0)] * 5


def test_one_step_of_k_stays_with_the_blocked_kernel(tmp_path):
    problems = [(kind, m, n, k_bytes, out) for kind in range(3) for out in (1, 2, 4) for m in (16, 32, 160, 1024) for n in (16, 128, 2048) for k_bytes in (32, 64, 128)]
    assert few_of(tmp_path, problems) == [(0, 0)] * len(problems)
