"""Wide waves of two runs of rows, which is how they lie where rows of a 32-bit D are 32 KiB apart: against one block per wave, exactly (small
whole numbers), and the same problem with rows of D a few elements further apart, which lies in one run."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_rungs import PAIRS, framed
from util import CM, RM
from wide_waves import RUNS_OF_ROWS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,pair,rung,m,n,k_bytes,out", RUNS_OF_ROWS)
def test_rows_of_d_32_kib_apart(kind, pair, rung, m, n, k_bytes, out):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k_bytes)
    la, lb = PAIRS[pair]
    k = k_bytes // (2 if kind == 0 else 1)
    result = torch.float32 if kind == 0 else torch.int32
    for dtype_in in ((orc.F16, orc.BF16) if kind == 0 else (orc.I8,)):
        dtype_out = orc.F32 if kind == 0 else orc.I32
        a, lda = framed(gen, dtype_in, *((m, k) if la == RM else (k, m)), -2, 2)
        b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
        c = torch.randint(-4, 5, (m + 1, n), generator=gen, device="cuda").to(result)
        bias = torch.randint(-8, 9, (n,), generator=gen, device="cuda").float()
        for beta in (0.0, -2.0):
            want = torch.empty((m, n), dtype=result, device="cuda")
            rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, want, 1.0, beta, lda=lda, ldb=ldb, algo=rw.GEMM_WAVE_TILE)
            for ldd in (n, n + 64):
                got = torch.full((m + 1, ldd), 77, dtype=result, device="cuda")
                rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, got, 1.0, beta, lda=lda, ldb=ldb, ldd=ldd)
                assert torch.equal(got[:m, :n], want), (dtype_in, beta, ldd)
                assert bool((got[m] == 77).all()) and bool((got[:, n:] == 77).all()), "wrote outside D"
                if kind == 0:
                    rw.gemm_bias_act(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, got, 1.0, beta, bias, rw.ACT_RELU, lda=lda, ldb=ldb, ldd=ldd)
                    assert torch.equal(got[:m, :n], torch.relu(want + bias)), (dtype_in, beta, ldd, "fused")
