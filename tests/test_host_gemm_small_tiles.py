"""The problems of tests/gemm_small_tiles.py run on the rungs they name, with the routes in front of the blocked GEMM asked as well (plain g++, no
GPU)."""
import os
import subprocess

import pytest

from gemm_small_tiles import CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def route_of(tmp_path_factory):
    exe = tmp_path_factory.mktemp("routes") / "route_of"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), os.path.join(ROOT, "tests", "host", "route_of.cpp")])
    return lambda text: subprocess.run([str(exe)], input=text, stdout=subprocess.PIPE, text=True, check=True).stdout.split("\n")


def test_cases_run_on_the_rungs_they_name(route_of):
    size = (2, 1, 1)
    asked = "".join(f"{kind} {pair} {m} {n} {k * size[kind]} {out}\n" for kind, pair, _, m, n, k, out in CASES)
    wrong = [(case, route) for case, route in zip(CASES, route_of(asked)) if case[2] != route]
    assert not wrong, wrong
