"""256 x 128 tiles on four waves where their ring of copies begins and wraps, against one block per wave (GEMM_WAVE_TILE): whole numbers as
operands, so that results must be equal bit for bit; the operands lie in frames of NaN (int8: 99), D in a guard."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_rungs import PAIRS, framed, guarded
from util import CM, RM
from wide_waves import RING_STARTS

pytestmark = pytest.mark.gpu

RESULTS = {(0, 4): [(orc.F16, orc.F32), (orc.BF16, orc.F32)], (0, 2): [(orc.F16, orc.F16), (orc.BF16, orc.BF16)], (1, 4): [(orc.I8, orc.I32)],
           (1, 1): [(orc.I8, orc.I8)]}


@pytest.mark.parametrize("kind,pair,rung,m,n,k_bytes,out", RING_STARTS)
def test_256_x_128_tiles_over_their_first_stages(kind, pair, rung, m, n, k_bytes, out):
    """256 x 128 tiles, whole and partly filled, where their ring (three stages of A, four of B) begins and wraps
    (tests/test_host_gemm_wide_waves.py says that these problems run on them)."""
    import torch

    gen = torch.Generator(device="cuda").manual_seed(k_bytes)
    la, lb = PAIRS[pair]
    for dtype_in, dtype_out in RESULTS[kind, out]:
        k = k_bytes // (1 if dtype_in == orc.I8 else 2)
        a, lda = framed(gen, dtype_in, m, k, -2, 2)
        b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        for alpha, beta in [(1.0, 0.0), (1.0, 1.0)]:
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            for d, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
                rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, d[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=algo)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta)
