"""The kernel whose waves share K (tests/few_rows.py) against one block per wave (GEMM_WAVE_TILE, itself compared with the oracle in
tests/test_gpu_gemm.py).  The operands are small whole numbers: products and sums are exact in whatever order, so results must be
equal bit for bit; the operands lie in frames of NaN (int8: 99), D in a guard."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from few_rows import CASES
from test_gpu_gemm_rungs import TYPES, framed, guarded, torch_type
from util import CM, RM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,mb,nb,m,n,k_bytes,out", CASES)
def test_few_rows_equal_one_block_per_wave(kind, mb, nb, m, n, k_bytes, out):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k_bytes)
    k = k_bytes // (2 if kind == 0 else 1)
    for dtype_in, dtype_out in TYPES[kind, out]:
        a, lda = framed(gen, dtype_in, m, k, -2, 2)
        b, ldb = framed(gen, dtype_in, n, k, -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        bias = torch.randint(-8, 9, (n,), generator=gen, device="cuda").float()
        for alpha, beta in [(1.0, 0.0), (2.0, -1.0)]:
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            for d, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
                rw.gemm(dtype_in, dtype_out, RM, CM, RM, m, n, k, a, b, c, d[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=algo)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta)
            if dtype_in == orc.I8:
                continue
            fused, plain, c32 = guarded(dtype_out, m, n), guarded(orc.F32, m, n), c.float()
            rw.gemm_bias_act(dtype_in, dtype_out, RM, CM, RM, m, n, k, a, b, c, fused[1024:], alpha, beta, bias, rw.ACT_RELU, lda=lda, ldb=ldb, ldc=ldc)
            rw.gemm(dtype_in, orc.F32, RM, CM, RM, m, n, k, a, b, c32, plain[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=rw.GEMM_WAVE_TILE)
            want = guarded(dtype_out, m, n)
            want[1024:1024 + m * n] = torch.relu(plain[1024:1024 + m * n].view(m, n) + bias).to(torch_type(dtype_out)).view(-1)
            assert torch.equal(fused.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta, "fused")
