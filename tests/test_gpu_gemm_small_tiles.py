"""The smallest tiles of the blocked GEMM on problems that run on them (tests/gemm_small_tiles.py), against one block per wave."""
import pytest

import test_gpu_gemm_rungs as rungs
from gemm_small_tiles import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,pair,rung,m,n,k,out", CASES)
def test_small_tiles_equal_one_block_per_wave(kind, pair, rung, m, n, k, out):
    rungs.test_rung_equals_one_block_per_wave(kind, pair, rung, m, n, k, out)
