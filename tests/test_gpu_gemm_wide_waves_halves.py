"""256 x 256 tiles whose last round runs as half tiles of 256 x 128 (four waves of 128 x 64 results, two stages of A and three of B), with and
without C, plain and with the fused epilogue: against one block per wave, exactly (small whole numbers)."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_rungs import PAIRS, framed, guarded, torch_type
from test_gpu_gemm_wide_waves_ring import RESULTS
from util import CM, RM
from wide_waves import HALF_TILES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,pair,rung,m,n,k_bytes,out", HALF_TILES)
def test_half_tiles_of_the_last_round(kind, pair, rung, m, n, k_bytes, out):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k_bytes)
    la, lb = PAIRS[pair]
    k = k_bytes // (2 if kind == 0 else 1)
    for dtype_in, dtype_out in RESULTS[kind, out]:
        a, lda = framed(gen, dtype_in, *((m, k) if la == RM else (k, m)), -2, 2)
        b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        for alpha, beta in [(1.0, 0.0), (2.0, -1.0)]:
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            for d, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
                rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, d[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=algo)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta)
            if dtype_in == orc.I8:
                continue
            bias = torch.randint(-8, 9, (n,), generator=gen, device="cuda").float()
            fused, plain, c32 = guarded(dtype_out, m, n), guarded(orc.F32, m, n), c.float()
            rw.gemm_bias_act(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, fused[1024:], alpha, beta, bias, rw.ACT_RELU, lda=lda, ldb=ldb, ldc=ldc)
            rw.gemm(dtype_in, orc.F32, la, lb, RM, m, n, k, a, b, c32, plain[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=rw.GEMM_WAVE_TILE)
            want = guarded(dtype_out, m, n)
            want[1024:1024 + m * n] = torch.relu(plain[1024:1024 + m * n].view(m, n) + bias).to(torch_type(dtype_out)).view(-1)
            assert torch.equal(fused.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta, "fused")
