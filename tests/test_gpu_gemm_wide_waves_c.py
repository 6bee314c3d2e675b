"""C and D in 16 and 8 bits on wide waves, which have all of their C in flight before the first result is stored: the same buffer as C and D,
plain and with the fused epilogue, against one block per wave, exactly (small whole numbers); C lies in a frame of NaN (int8: 99)."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_rungs import PAIRS, TYPES, framed, torch_type
from util import CM, RM
from wide_waves import NARROW_C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,pair,rung,m,n,k_bytes,out", NARROW_C)
def test_c_in_place(kind, pair, rung, m, n, k_bytes, out):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k_bytes)
    la, lb = PAIRS[pair]
    k = k_bytes // (2 if kind == 0 else 1)
    for dtype_in, dtype_out in TYPES[kind, out]:
        a, lda = framed(gen, dtype_in, *((m, k) if la == RM else (k, m)), -2, 2)
        b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        got, want = c.clone(), c.clone()
        for d, algo in ((got, rw.GEMM_AUTO), (want, rw.GEMM_WAVE_TILE)):
            rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, d, d, 1.0, -2.0, lda=lda, ldb=ldb, ldc=ldc, ldd=ldc, algo=algo)
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out)
        if dtype_in == orc.I8:
            continue
        bias = torch.randint(-8, 9, (n,), generator=gen, device="cuda").float()
        got, plain, c32 = c.clone(), torch.empty((m, ldc), device="cuda"), c.float()
        rw.gemm_bias_act(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, got, got, 1.0, -2.0, bias, rw.ACT_RELU, lda=lda, ldb=ldb, ldc=ldc, ldd=ldc)
        rw.gemm(dtype_in, orc.F32, la, lb, RM, m, n, k, a, b, c32, plain, 1.0, -2.0, lda=lda, ldb=ldb, ldc=ldc, ldd=ldc, algo=rw.GEMM_WAVE_TILE)
        want = c.clone()
        want[:m, :n] = torch.relu(plain[:, :n] + bias).to(torch_type(dtype_out))
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, "fused")
