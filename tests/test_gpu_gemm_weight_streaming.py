"""The weight-streaming kernel that has all of A in LDS (tests/weight_streaming.py) against one block per wave (GEMM_WAVE_TILE, itself compared
with the oracle in tests/test_gpu_gemm.py): whole numbers as operands, so that results must be equal bit for bit; the operands lie in
frames of NaN (int8: 99), D in a guard."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_rungs import framed, guarded
from util import CM, RM
from weight_streaming import CASES

pytestmark = pytest.mark.gpu

TYPES = {0: [(orc.F16, orc.F32), (orc.BF16, orc.F32)], 1: [(orc.I8, orc.I32)], 2: [(orc.E4M3, orc.F32), (orc.E5M2, orc.F32)]}


@pytest.mark.parametrize("kind,steps,m,n,k_bytes", CASES)
def test_weight_streaming_equals_one_block_per_wave(kind, steps, m, n, k_bytes):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k_bytes)
    k = k_bytes // (2 if kind == 0 else 1)
    for dtype_in, dtype_out in TYPES[kind]:
        a, lda = framed(gen, dtype_in, m, k, -2, 2)
        b, ldb = framed(gen, dtype_in, n, k, -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        for alpha, beta in [(1.0, 0.0), (2.0, -3.0)]:
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            for d, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
                rw.gemm(dtype_in, dtype_out, RM, CM, RM, m, n, k, a, b, c, d[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=algo)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, beta)
        # the same buffer as C and D
        got, want = c.clone(), c.clone()
        for d, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
            rw.gemm(dtype_in, dtype_out, RM, CM, RM, m, n, k, a, b, d, d, 2.0, -3.0, lda=lda, ldb=ldb, ldc=ldc, ldd=ldc, algo=algo)
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, "in place")
