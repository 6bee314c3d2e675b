"""Both weight-streaming kernels on problems that run on them: against the oracle on operands that are no whole numbers, and replayed from
a graph.  All of A in LDS beyond 8192 columns, slices of K over workgroups for up to 48 rows and more than 4 KiB of K
(tests/test_host_gemm_weight_streaming.py says that these problems run there)."""
import pytest

import oracle as orc
import rocwmma_amd as rw
import test_gpu_gemm as plain
import test_gpu_graph_replay as replays
from weight_streaming import HALF, REPLAYED, SLICED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("route,m,n,k", HALF)
@pytest.mark.parametrize("dtype_in", [orc.F16, orc.BF16])
def test_16_bit(dtype_in, route, m, n, k):
    plain.test_skinny_and_sliced_kernels_16bit(dtype_in, m, n, k)


@pytest.mark.parametrize("m,n,k", SLICED)
@pytest.mark.parametrize("dtype_in", [orc.I8, orc.E4M3, orc.E5M2])
def test_slices_of_k(dtype_in, m, n, k):
    plain.test_sliced_weight_streaming_kernel(dtype_in, m, n, k)


@pytest.mark.parametrize("kind,route,m,n,k", REPLAYED)
def test_replays(kind, route, m, n, k):
    dtype_in, dtype_out = (orc.I8, orc.I32) if kind == 1 else (orc.E4M3, orc.F32)
    replays.test_gemm_replays(dtype_in, dtype_out, m, n, k, rw.GEMM_AUTO)
