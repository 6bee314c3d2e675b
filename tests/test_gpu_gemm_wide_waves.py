"""The 256 x 256 tile's loop (GEMM_BLOCKED_256) over its first stage counts, where a ring of two stages of A and three of B begins, wraps
and ends: against one block per wave, exactly (small whole numbers)."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_rungs import PAIRS, framed, guarded
from util import CM, RM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 6, 13])
@pytest.mark.parametrize("dtype_in,dtype_out", [(orc.F16, orc.F32), (orc.BF16, orc.BF16), (orc.I8, orc.I32), (orc.I8, orc.I8)])
def test_every_stage_count(dtype_in, dtype_out, stages):
    import torch

    m, n, k = 512, 768, stages * (128 if dtype_in == orc.I8 else 64)
    gen = torch.Generator(device="cuda").manual_seed(stages)
    for la, lb in PAIRS:
        a, lda = framed(gen, dtype_in, *((m, k) if la == RM else (k, m)), -2, 2)
        b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        for alpha, beta in [(1.0, 0.0), (2.0, -1.0)]:
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            for out, algo in ((got, rw.GEMM_BLOCKED_256), (want, rw.GEMM_WAVE_TILE)):
                rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, out[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=algo)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (la, lb, beta)


@pytest.mark.parametrize("m,n", [(1536, 3584), (528, 7184), (1040, 6000)])
@pytest.mark.parametrize("k_bytes", [256, 384, 512, 640, 768, 1312, 2080])
def test_halves_over_their_first_stages(k_bytes, m, n):
    """256 x 128 tiles, whole and partly filled, where their ring (three stages of A, four of B) begins and wraps."""
    import torch

    gen = torch.Generator(device="cuda").manual_seed(k_bytes)
    for dtype_in, dtype_out in [(orc.F16, orc.F16), (orc.BF16, orc.F32), (orc.I8, orc.I32)]:
        k = k_bytes // (1 if dtype_in == orc.I8 else 2)
        for lb in (CM, RM):
            a, lda = framed(gen, dtype_in, m, k, -2, 2)
            b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
            c, ldc = framed(gen, dtype_out, m, n, -4, 4)
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            for out, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
                rw.gemm(dtype_in, dtype_out, RM, lb, RM, m, n, k, a, b, c, out[1024:], 1.0, 1.0, lda=lda, ldb=ldb, ldc=ldc, algo=algo)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, lb)
