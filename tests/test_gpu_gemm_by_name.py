"""K of the blocked GEMM asked for by name: whole 64-byte stages, three of them, or two where the problem is more than one
round of workgroups (or the 256 x 256 tile is named)."""
import numpy as np
import pytest

import oracle as orc
import rocwmma_amd as rw
from util import CM, RM, exact_int_bits, to_device, to_host

pytestmark = pytest.mark.gpu

# (algo, m, n, layout of B, K bytes, taken on 256 compute units)
CASES = [(rw.GEMM_BLOCKED_256, 256, 256, CM, 128, True), (rw.GEMM_BLOCKED_256, 256, 512, RM, 128, True), (rw.GEMM_BLOCKED_256, 256, 256, CM, 192, False),
         (rw.GEMM_BLOCKED_256, 256, 256, CM, 64, False), (rw.GEMM_BLOCKED, 256, 256, CM, 128, False), (rw.GEMM_BLOCKED, 256, 256, RM, 192, True),
         (rw.GEMM_BLOCKED, 2816, 3072, CM, 128, True), (rw.GEMM_BLOCKED, 2816, 3072, RM, 128, True), (rw.GEMM_BLOCKED, 1088, 1088, CM, 128, True),
         (rw.GEMM_BLOCKED, 1088, 1088, RM, 128, False), (rw.GEMM_BLOCKED, 1040, 1040, CM, 128, False), (rw.GEMM_BLOCKED, 2064, 2064, CM, 128, True),
         (rw.GEMM_BLOCKED, 2064, 2064, RM, 128, True), (rw.GEMM_BLOCKED, 2816, 3072, CM, 96, False), (rw.GEMM_BLOCKED, 2816, 3072, CM, 64, False)]


@pytest.mark.parametrize("dtype_in,dtype_out", [(orc.F16, orc.F32), (orc.I8, orc.I32), (orc.E4M3, orc.F32)])
@pytest.mark.parametrize("algo,m,n,lb,kbytes,taken", CASES)
def test_shortest_k_by_name(dtype_in, dtype_out, algo, m, n, lb, kbytes, taken):
    import torch

    if rw.device_info()["compute_units"] != 256:
        pytest.skip("the rule goes by the compute units")
    k = kbytes // (2 if dtype_in == orc.F16 else 1)
    a, b = exact_int_bits(dtype_in, m, k, RM), exact_int_bits(dtype_in, k, n, lb)
    d = to_device(np.full(m * n, 77, dtype=orc.storage_dtype(dtype_out)))
    call = lambda which: rw.gemm(dtype_in, dtype_out, RM, lb, RM, m, n, k, to_device(a), to_device(b), None, d, 1.0, 0.0, algo=which)
    if not taken:
        with pytest.raises(rw.RocwmmaError) as err:
            call(algo)
        assert err.value.status == 3  # unsupported shape
        return
    call(algo)
    torch.cuda.synchronize()
    want = orc.gemm(dtype_in, dtype_out, RM, lb, RM, RM, m, n, k, a, b, None, 1.0, 0.0)
    assert np.array_equal(to_host(d, orc.storage_dtype(dtype_out)), want)
