"""Leading dimensions so large that the rows of a tile, or of a stage of K, span more than the 2 GiB window its copies address: the
smaller tiles and the 64-byte stages take those, by name and chosen by the library; beyond them the call is refused.  Whole
numbers as operands: exact results."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from util import CM, RM

pytestmark = pytest.mark.gpu

MB = 1 << 20
# (layouts of A and B, m, n, k, bytes between A's rows (row-major) or columns, taken): 128 rows, 64 rows and 32 K rows of that pitch
# are below 2 GiB, or none of them
CASES = [(RM, CM, 64, 1040, 192, 15 * MB, True), (RM, CM, 64, 1040, 192, 17 * MB, True), (RM, CM, 64, 272, 96, 31 * MB, True),
         (CM, CM, 160, 48, 96, 31 * MB, True), (CM, CM, 160, 48, 96, 34 * MB, True), (CM, CM, 272, 64, 96, 63 * MB, True), (CM, RM, 144, 272, 96, 34 * MB, True),
         (CM, RM, 144, 272, 80, 63 * MB, True), (CM, RM, 144, 272, 64, 68 * MB, False)]


@pytest.mark.parametrize("la,lb,m,n,k,pitch,taken", CASES)
@pytest.mark.parametrize("algo", [rw.GEMM_AUTO, rw.GEMM_BLOCKED])
def test_wide_rows(algo, la, lb, m, n, k, pitch, taken):
    import torch

    if algo == rw.GEMM_BLOCKED and taken and (k * 2 % 64 or k * 2 < 192):
        pytest.skip("three whole 64-byte stages by name")
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    whole = lambda *shape: torch.randint(-2, 3, shape, generator=gen, device="cuda").half()
    rows, cols = (m, k) if la == RM else (k, m)
    lda = pitch // 2
    big = torch.empty((rows - 1) * lda + cols, dtype=torch.float16, device="cuda")
    a = torch.as_strided(big, (rows, cols), (lda, 1))
    a.copy_(whole(rows, cols))
    b = whole(*((n, k) if lb == CM else (k, n)))
    d = torch.full((m, n), 77.0, device="cuda")
    call = lambda: rw.gemm(orc.F16, orc.F32, la, lb, RM, m, n, k, big, b, None, d, 1.0, 0.0, lda=lda, algo=algo)
    if not taken:
        with pytest.raises(rw.RocwmmaError) as err:
            call()
        assert err.value.status == 3  # unsupported shape
        return
    call()
    wa = a.contiguous().float() if la == RM else a.t().contiguous().float()
    wb = b.t().contiguous().float() if lb == CM else b.float()
    assert torch.equal(d, wa @ wb)
