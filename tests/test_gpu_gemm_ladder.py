"""The blocked GEMM on sizes that fill neither tiles nor K stages, one block to the largest tiles: K shorter than the
pipeline's prologue and ending inside a stage, all element types, plain and with the fused epilogue.  (Which of the tiles and
pipelines a size runs on is for the cost table to say; tests/test_gpu_gemm_rungs.py reaches every one of them by name.)

Operands are padded (leading dimensions and further K rows) with NaN (int8: 99), so a copy that reads past the
end of K or lets a padded byte into a sum shows in the result; D is framed by a guard.  The oracle sees the same bits
without the padding.  Tolerances: those of tests/test_gpu_gemm.py; float32: partial sums of k products of values
uniform in [-1, 1] are about sqrt(k) / 3, their k roundings of 2^-24 add up as a random walk to k / 3 * 2^-24 on
either side, so twice that."""
import numpy as np
import pytest

import oracle as orc
import rocwmma_amd as rw
from util import CM, RM, normal_fp8_bits, to_device, to_host, tol_for, uniform_bits

pytestmark = pytest.mark.gpu

# (m, n, k): one tile with K below one stage; 64-, 128 x 64- and 128-wide tiles; 256 x 128; 256 x 256; few rows, many columns
SHAPES = [(16, 16, 32), (48, 272, 32), (272, 400, 1056), (1040, 1104, 608), (208, 10256, 480), (2000, 3056, 352), (3600, 3856, 224)]
PAIRS = [(RM, CM), (RM, RM), (CM, CM), (CM, RM)]


def padded(bits, dtype, rows, cols, pad):
    """rows x cols (cols contiguous) in a frame of `pad` more columns and 64 more rows of NaN."""
    if dtype == orc.F32:
        poison = np.float32(np.nan)
    else:
        poison = {orc.F16: 0x7E00, orc.BF16: 0x7FC0, orc.E4M3: 0x7F, orc.E5M2: 0x7F, orc.I8: 99}[dtype]
    big = np.full((rows + 64, cols + pad), poison, dtype=bits.dtype)
    big[:rows, :cols] = bits.reshape(rows, cols)
    return to_device(big.ravel()), cols + pad


def bits_for(seed, dtype, count):
    if dtype in (orc.E4M3, orc.E5M2):
        return normal_fp8_bits(seed, dtype, count)
    if dtype == orc.I8:
        return np.random.default_rng(seed).integers(-9, 10, count, dtype=np.int8)
    return uniform_bits(seed, dtype, count)


def operands(dtype, la, lb, m, n, k):
    size = {orc.F32: 4, orc.F16: 2, orc.BF16: 2}.get(dtype, 1)
    pad = 48 // size
    a, b = bits_for(m + k, dtype, m * k), bits_for(n + k + 1, dtype, k * n)
    da, lda = padded(a, dtype, *((m, k) if la == RM else (k, m)), pad)
    db, ldb = padded(b, dtype, *((n, k) if lb == CM else (k, n)), pad)
    return a, b, da, lda, db, ldb


def framed(dtype_out, count):
    guard = 4096
    frame = np.zeros(count + 2 * guard, dtype=orc.storage_dtype(dtype_out))
    frame[:] = 12345.0 if frame.dtype == np.float32 else 0x55
    dev = to_device(frame)
    return frame, dev, dev[guard:guard + count]


def compare(dtype_in, dtype_out, frame, dev, want, tol):
    guard = 4096
    host = to_host(dev, frame.dtype)
    assert np.array_equal(host[:guard], frame[:guard]) and np.array_equal(host[-guard:], frame[-guard:]), "wrote outside D"
    got = np.ascontiguousarray(host[guard:-guard])
    if tol == 0.0:
        assert np.array_equal(got, want), f"{(got != want).sum()} of {got.size} elements differ"
        return
    err, inf, nan = orc.compare_equal(dtype_out, got, dtype_out, want)
    assert not inf and not nan and err <= tol, (err, inf, nan)


@pytest.mark.parametrize("la,lb", PAIRS)
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dtype_in,dtype_out", [(orc.F16, orc.F32), (orc.BF16, orc.BF16), (orc.I8, orc.I32), (orc.I8, orc.I8),
                                                (orc.E4M3, orc.F32), (orc.E5M2, orc.F32), (orc.F32, orc.F32)])
def test_partly_filled_tiles_and_stages(dtype_in, dtype_out, m, n, k, la, lb):
    import torch

    if m * n > 1 << 23 and dtype_in in (orc.E5M2, orc.BF16):
        pytest.skip("the largest tile: one type per element size")
    if dtype_in in (orc.F16, orc.BF16):
        k += 16  # (an odd number of 32-byte pieces)
    a, b, da, lda, db, ldb = operands(dtype_in, la, lb, m, n, k)
    c = uniform_bits(7, dtype_out, m * n) if dtype_out != orc.I8 else bits_for(7, orc.I8, m * n)
    tol = 4e-3 if dtype_out == orc.BF16 else 2.0 * k / 3.0 * 2.0 ** -24 if dtype_in == orc.F32 else tol_for(dtype_in)
    for lc, beta in [(RM, 0.0), (RM, -1.0), (CM, 2.0)]:
        if lc == CM and m * n > 1 << 21:
            continue  # (the transposed problem on the same kernels)
        frame, dev, d = framed(dtype_out, m * n)
        rw.gemm(dtype_in, dtype_out, la, lb, lc, m, n, k, da, db, to_device(c), d, 1.0, beta, lda=lda, ldb=ldb)
        torch.cuda.synchronize()
        want = orc.gemm(dtype_in, dtype_out, la, lb, lc, lc, m, n, k, a, b, c, 1.0, beta)
        compare(dtype_in, dtype_out, frame, dev, want, tol)


@pytest.mark.parametrize("la,lb", PAIRS)
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dtype_in,dtype_out", [(orc.F16, orc.F16), (orc.BF16, orc.F32), (orc.E4M3, orc.F32)])
def test_fused_epilogue_on_every_rung(dtype_in, dtype_out, m, n, k, la, lb):
    import torch

    if dtype_in != orc.E4M3:
        k += 16
    a, b, da, lda, db, ldb = operands(dtype_in, la, lb, m, n, k)
    c = uniform_bits(8, dtype_out, m * n)
    bias = np.random.default_rng(9).uniform(-1, 1, n).astype(np.float32)
    for act, beta in [(rw.ACT_GELU, 0.0), (rw.ACT_RELU, 1.0)]:
        frame, dev, d = framed(dtype_out, m * n)
        rw.gemm_bias_act(dtype_in, dtype_out, la, lb, RM, m, n, k, da, db, to_device(c), d, 1.0, beta, to_device(bias), act, lda=lda, ldb=ldb)
        torch.cuda.synchronize()
        want = orc.gemm_bias_act(dtype_in, dtype_out, la, lb, RM, m, n, k, a, b, c, 1.0, beta, bias, act)
        compare(dtype_in, dtype_out, frame, dev, want, tol_for(dtype_in))
