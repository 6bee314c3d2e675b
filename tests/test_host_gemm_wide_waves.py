"""The problems of tests/wide_waves.py run on the rungs they name (plain g++, no GPU)."""
import pytest

import wide_waves
from test_host_gemm_small_tiles import route_of  # noqa: F401  (the fixture)


@pytest.mark.parametrize("name", [name for name in dir(wide_waves) if name.isupper()])
def test_cases_run_on_the_rungs_they_name(route_of, name):  # noqa: F811
    cases = getattr(wide_waves, name)
    asked = "".join("%d %d %d %d %d %d\n" % (kind, pair, m, n, k_bytes, out) for kind, pair, _, m, n, k_bytes, out in cases)
    wrong = [(case, rung) for case, rung in zip(cases, route_of(asked)) if case[2] != rung]
    assert not wrong, wrong


def test_half_tiles_have_a_last_round_of_at_most_half_the_units():
    for kind, pair, rung, m, n, k_bytes, out in wide_waves.HALF_TILES:
        assert m % 256 == 0 and n % 256 == 0 and k_bytes % 128 == 0
        tiles = (m // 256) * (n // 256)
        assert tiles > 256 and 0 < tiles % 256 <= 128
