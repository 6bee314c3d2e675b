"""The problems of tests/weight_streaming.py run on the weight-streaming kernel, with as many K steps fetched together as they name, and where
its neighbours take over (plain g++, no GPU)."""
from test_host_gemm_small_tiles import route_of  # noqa: F401  (the fixture)
from weight_streaming import CASES, HALF, REPLAYED, SLICED


def test_cases_run_on_the_kernel_they_name(route_of):  # noqa: F811
    asked = "".join(f"{kind} 0 {m} {n} {k_bytes} 4\n" for kind, _, m, n, k_bytes in CASES)
    wrong = [(case, route) for case, route in zip(CASES, route_of(asked)) if route != f"Skinny{case[1]}"]
    assert not wrong, wrong


def test_cases_of_the_oracle_run_on_the_kernel_they_name(route_of):  # noqa: F811
    problems = [(f"0 0 {m} {n} {2 * k} 4\n", route) for route, m, n, k in HALF]
    problems += [(f"{kind} 0 {m} {n} {k} 4\n", "Sliced") for kind in (1, 2) for m, n, k in SLICED]
    problems += [(f"{kind} 0 {m} {n} {k} 4\n", route) for kind, route, m, n, k in REPLAYED]
    got = route_of("".join(asked for asked, _ in problems))
    wrong = [(problem, route) for problem, route in zip(problems, got) if problem[1] != route]
    assert not wrong, wrong


def test_neighbours(route_of):  # noqa: F811
    # 32 columns per unit; K in whole KiB; 32-bit results; 32 rows; A within 128 KiB of LDS, beyond it K slices for up to 48 rows, none
    # from 64 on
    for problem, route in [("1 0 16 8192 4096 4", "Few"), ("1 0 16 8208 4096 4", "Skinny8"), ("1 0 24 8208 4096 4", None),
                           ("0 0 16 8208 1536 4", None), ("0 0 16 8208 4096 2", None), ("1 0 32 8208 5120 4", None),
                           ("1 0 32 6656 5120 4", "Sliced"), ("1 0 48 5120 5120 4", "Sliced"), ("1 0 48 5136 5120 4", None),
                           ("1 0 64 5120 5120 4", None)]:
        got = route_of(problem + "\n")[0]
        assert got == route if route else not got.startswith(("Skinny", "Sliced")), (problem, got)
