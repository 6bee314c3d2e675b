"""Results rounded to bfloat16: to nearest, ties to even, past the largest finite value to infinity, NaN to NaN.  Every result is the exact
sum of three bfloat16 parts of a float32 value, so what is tested is the rounding alone."""
import pytest

import rocwmma_amd as rw

pytestmark = pytest.mark.gpu


def values(n):
    import torch

    gen = torch.Generator().manual_seed(5)
    v = torch.randn(n, generator=gen) * torch.exp2(torch.randint(-60, 61, (n,), generator=gen).float())
    bits = v.view(torch.int32)
    bits[0::4] = (bits[0::4] & ~0xFFFF) | 0x8000  # ties
    bits[1::8] = (bits[1::8] & ~0xFFFF) | 0x7FFF
    bits[2::8] = (bits[2::8] & ~0xFFFF) | 0x8001
    v[:4] = torch.tensor([0.0, -0.0, 3.3961775e38, -3.3961775e38])  # (the last two: halfway to 2^128, a tie that goes to infinity)
    return v


@pytest.mark.parametrize("algo,m,n", [(rw.GEMM_AUTO, 4096, 4096), (rw.GEMM_AUTO, 2000, 3056), (rw.GEMM_AUTO, 208, 80), (rw.GEMM_WAVE_TILE, 512, 256)])
def test_results_are_rounded_to_nearest_even(algo, m, n):
    import torch

    k = 512
    v = values(m)
    parts, rest = [], v.clone()
    for _ in range(3):
        p = (rest.view(torch.int32) & ~0xFFFF).view(torch.float32)
        parts.append(p)
        rest = rest - p
    a = torch.zeros((m, k))
    for i, p in enumerate(parts):
        a[:, i] = p
    special = torch.tensor([float("inf"), float("-inf"), float("nan")])
    a[4:7, 0] = special
    a[4:7, 1:3] = 0.0
    v[4:7] = special
    b = torch.zeros((n, k))
    b[:, :3] = 1.0
    a, b = a.to(torch.bfloat16).cuda(), b.to(torch.bfloat16).cuda()
    # (infinities and NaN meet the zeros of b as well: only in columns of a that are zero elsewhere)
    want = v.to(torch.bfloat16).cuda().view(m, 1).expand(m, n)
    d = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    c = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
    for beta in (0.0, 1.0):
        rw.gemm(rw.BF16, rw.BF16, rw.ROW_MAJOR, rw.COL_MAJOR, rw.ROW_MAJOR, m, n, k, a, b, c, d, 1.0, beta, algo=algo)
        assert torch.equal(d.isnan(), want.isnan())
        assert torch.equal(d.nan_to_num(7.0, float("inf"), float("-inf")), want.nan_to_num(7.0, float("inf"), float("-inf")))
