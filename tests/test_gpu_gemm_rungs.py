"""Every rung of the blocked GEMM (tests/gemm_rungs.py), plain and with the fused epilogue, against one block per wave
(GEMM_WAVE_TILE, itself compared with the oracle in tests/test_gpu_gemm.py).  The operands are small whole numbers, so that every
product and partial sum is exact in whatever order and the results must be equal bit for bit; they lie in frames of NaN (int8:
99), and D in a guard."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from gemm_rungs import CASES
from util import CM, RM

pytestmark = pytest.mark.gpu

PAIRS = [(RM, CM), (RM, RM), (CM, CM), (CM, RM)]
TYPES = {(0, 4): [(orc.F16, orc.F32), (orc.BF16, orc.F32), (orc.F16, orc.F16), (orc.BF16, orc.BF16)], (1, 4): [(orc.I8, orc.I32), (orc.I8, orc.I8)],
         (0, 2): [(orc.F16, orc.F16), (orc.BF16, orc.BF16)], (1, 1): [(orc.I8, orc.I8)], (2, 4): [(orc.E4M3, orc.F32), (orc.E5M2, orc.F32)]}


def torch_type(dtype):
    import torch

    return {orc.F16: torch.float16, orc.BF16: torch.bfloat16, orc.E4M3: torch.float8_e4m3fn, orc.E5M2: torch.float8_e5m2, orc.I8: torch.int8,
            orc.F32: torch.float32, orc.I32: torch.int32}[dtype]


def framed(gen, dtype, rows, cols, low, high):
    """rows x cols whole numbers in a frame of 48 more bytes per row and 64 more rows of NaN."""
    import torch

    size = torch.empty(0, dtype=torch_type(dtype)).element_size()
    ld = cols + 48 // size
    big = torch.full((rows + 64, ld), 99.0 if dtype in (orc.I8, orc.I32) else float("nan"), device="cuda")
    big[:rows, :cols] = torch.randint(low, high + 1, (rows, cols), generator=gen, device="cuda").float()
    return big.to(torch_type(dtype)), ld


def guarded(dtype, rows, cols):
    import torch

    return torch.full((rows * cols + 2048,), 77, dtype=torch.float32, device="cuda").to(torch_type(dtype))


@pytest.mark.parametrize("kind,pair,rung,m,n,k,out", CASES)
def test_rung_equals_one_block_per_wave(kind, pair, rung, m, n, k, out):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    la, lb = PAIRS[pair]
    for dtype_in, dtype_out in TYPES[kind, out]:
        a, lda = framed(gen, dtype_in, *((m, k) if la == RM else (k, m)), -2, 2)
        b, ldb = framed(gen, dtype_in, *((n, k) if lb == CM else (k, n)), -2, 2)
        c, ldc = framed(gen, dtype_out, m, n, -4, 4)
        bias = torch.randint(-8, 9, (n,), generator=gen, device="cuda").float()
        for alpha, beta in [(1.0, 0.0), (1.0, -2.0)]:
            got, want = guarded(dtype_out, m, n), guarded(dtype_out, m, n)
            rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, got[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc)
            rw.gemm(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, want[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=rw.GEMM_WAVE_TILE)
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta)
            if dtype_in == orc.I8:
                continue
            # (the bias and ReLU of whole numbers are exact as well; a result of 16 bits is rounded once on either side)
            fused = guarded(dtype_out, m, n)
            rw.gemm_bias_act(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, fused[1024:], alpha, beta, bias, rw.ACT_RELU, lda=lda, ldb=ldb, ldc=ldc)
            plain = guarded(orc.F32, m, n)
            c32 = c.float()
            rw.gemm(dtype_in, orc.F32, la, lb, RM, m, n, k, a, b, c32, plain[1024:], alpha, beta, lda=lda, ldb=ldb, ldc=ldc, algo=rw.GEMM_WAVE_TILE)
            want = guarded(dtype_out, m, n)
            want[1024:1024 + m * n] = torch.relu(plain[1024:1024 + m * n].view(m, n) + bias).to(torch_type(dtype_out)).view(-1)
            assert torch.equal(fused.view(torch.uint8), want.view(torch.uint8)), (dtype_in, dtype_out, beta, "fused")
