"""Few token rows on either side of the rule that hands them from the K-sliced weight-streaming kernel (two launches: D = beta * C,
then atomic adds of the slices) to the blocked kernel (one launch).  Whole numbers as operands: exact results in any order."""
import pytest

import oracle as orc
import rocwmma_amd as rw
from test_gpu_gemm_mx_raw import launches_of
from util import CM, RM

pytestmark = pytest.mark.gpu

# (m, n, bytes of K, sliced on 256 compute units): 4 KiB of K, columns per KiB of K, 32 columns per unit, A of 16 / 32 rows beyond the
# LDS, remainders of the 256 columns of a workgroup
CASES = [(48, 272, 4096, False), (48, 16, 5120, True), (48, 5120, 5120, True), (48, 5136, 5120, False), (48, 6144, 6144, True),
         (48, 6160, 6144, False), (48, 8192, 8192, True), (48, 8208, 8192, False), (48, 1040, 29696, True), (32, 6656, 5120, True),
         (32, 6672, 5120, False), (32, 8192, 6144, True), (32, 8208, 6144, False), (16, 8192, 9216, True), (16, 8208, 9216, False)]


@pytest.mark.parametrize("dtype_in,dtype_out", [(orc.F16, orc.F32), (orc.BF16, orc.F32), (orc.I8, orc.I32), (orc.E4M3, orc.F32)])
@pytest.mark.parametrize("m,n,kbytes,sliced", CASES)
def test_either_side_of_the_rule(dtype_in, dtype_out, m, n, kbytes, sliced):
    import torch

    if rw.device_info()["compute_units"] != 256:
        pytest.skip("the rule goes by the compute units")
    storage = {orc.F16: torch.float16, orc.BF16: torch.bfloat16, orc.I8: torch.int8, orc.E4M3: torch.float8_e4m3fn}[dtype_in]
    result = torch.int32 if dtype_in == orc.I8 else torch.float32
    k = kbytes // storage.itemsize
    gen = torch.Generator(device="cuda").manual_seed(m + n + kbytes)
    whole = lambda *shape: torch.randint(-2, 3, shape, generator=gen, device="cuda")
    a, b, c = whole(m, k), whole(n, k), whole(m, n)
    d = torch.full((m, n), 77, device="cuda", dtype=result)
    da, db, dc = a.float().to(storage), b.float().to(storage), c.to(result)
    call = lambda: rw.gemm(dtype_in, dtype_out, RM, CM, RM, m, n, k, da, db, dc, d, 2.0, 3.0)
    call()
    torch.cuda.synchronize()
    # (sums below 2^24)
    want = 2 * (a.float() @ b.t().contiguous().float()) + 3 * c.float()
    assert torch.equal(d.float(), want)
    assert launches_of(call) == (2 if sliced else 1)
