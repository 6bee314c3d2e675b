"""Which rung of the blocked GEMM a problem runs on (plain g++, no GPU): the problems of tests/gemm_rungs.py reach every rung that
there is, partly filled and whole."""
import os
import subprocess

import pytest

from gemm_rungs import CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rung_of(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rungs") / "rung_of"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), os.path.join(ROOT, "tests", "host", "rung_of.cpp")])
    return lambda *args, text="": subprocess.run([str(exe), *args], input=text, stdout=subprocess.PIPE, text=True, check=True).stdout.split("\n")


def test_cases_run_on_the_rungs_they_name(rung_of):
    size = (2, 1, 1)
    asked = "".join(f"{kind} {pair} {m} {n} {k * size[kind]} {out}\n" for kind, pair, _, m, n, k, out in CASES)
    got = rung_of(text=asked)
    wrong = [(case, rung) for case, rung in zip(CASES, got) if case[2] != rung]
    assert not wrong, wrong


def test_every_rung_has_a_partly_filled_and_a_whole_case(rung_of):
    size = (2, 1, 1)
    rungs = {(int(a), int(b), c) for a, b, c in (line.split() for line in rung_of("rungs") if line)}
    whole = {case[:3] for case in CASES if case[3] % 128 == 0 and case[4] % 128 == 0 and case[5] * size[case[0]] % 128 == 0}
    edges = {case[:3] for case in CASES if case[3] % 64 and case[4] % 64 and case[5] * size[case[0]] % 64}
    # (what is never chosen, partly filled or whole, is there for operands that larger tiles cannot address)
    assert rungs - whole == {(1, 2, "Ring4"), (1, 3, "Mid")}
    assert rungs - edges == {(1, 0, "NarrowLines")}
    # (one block per wave is no tile of the blocked kernel: short K only)
    assert edges - rungs == {(kind, pair, "WaveTile") for kind in range(3) for pair in range(4)}
