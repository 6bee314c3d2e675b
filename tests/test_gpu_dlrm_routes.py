"""DLRM sizes on either side of the rules that choose between the kernels (whole small samples, samples in LDS, tiles), by
batch, rows and width on 256 compute units, against the CPU oracle; a sample of NaNs between the others must not reach them.
Tolerances as in tests/test_gpu_dlrm_sample.py."""
import numpy as np
import pytest

import oracle as orc
import rocwmma_amd as rw
from util import to_device, uniform_bits

pytestmark = pytest.mark.gpu

# (dtype, batch, m, k): up to 32 rows of the usual widths, by batch and by rows; width 32 backward; float16 samples of more than half
# the LDS; few float32 samples of more than 160 rows; wide float32 samples backward
BOTH = [(orc.F16, 1, 1, 32), (orc.F16, 7, 16, 64), (orc.F16, 5, 8, 128), (orc.F16, 3, 32, 256), (orc.F16, 5, 3, 256), (orc.F16, 512, 27, 256),
        (orc.F16, 513, 27, 256), (orc.F16, 4096, 13, 32), (orc.F16, 4097, 13, 32), (orc.F16, 2047, 27, 32), (orc.F16, 2048, 29, 32),
        (orc.F16, 256, 96, 512), (orc.F16, 257, 96, 512), (orc.F16, 85, 192, 256), (orc.F16, 86, 192, 256), (orc.F32, 85, 161, 64),
        (orc.F32, 86, 161, 64), (orc.F32, 3, 160, 64), (orc.F32, 2, 192, 136), (orc.F32, 85, 40, 264), (orc.F32, 86, 40, 264), (orc.F32, 2, 64, 516)]
# forward only: many rounds of tiles of a few rows of tiles
FORWARD = [(orc.F16, 2047, 193, 8), (orc.F16, 2048, 193, 8), (orc.F16, 2048, 250, 16), (orc.F16, 511, 300, 24), (orc.F16, 512, 300, 24),
           (orc.F16, 512, 352, 8), (orc.F16, 512, 353, 8), (orc.F16, 1229, 400, 8)]


def poison(bits, sample, nan):
    out = bits.copy()
    out[sample] = nan
    return out


@pytest.mark.parametrize("dtype,batch,m,k,backward", [(*c, True) for c in BOTH] + [(*c, False) for c in FORWARD])
def test_either_side_of_the_rules(dtype, batch, m, k, backward):
    import torch

    np_t, nan = (np.uint16, 0x7E00) if dtype == orc.F16 else (np.float32, np.nan)
    width = k + m * (m - 1) // 2
    feat = uniform_bits(m + k, dtype, batch * m * k).reshape(batch, m * k)
    poisoned = batch // 2 if batch > 1 else -1
    bad = lambda bits: poison(bits, poisoned, nan) if poisoned >= 0 else bits
    dev_feat = to_device(bad(feat).ravel())
    out = to_device(np.full(batch * width, nan, dtype=np_t))
    rw.dlrm_fwd(dev_feat, out, m, k, batch, dtype)
    # the oracle takes the first and last samples, the poisoned one's neighbours and some between
    keep = sorted(({0, 1, 2, 3, batch - 2, batch - 1, batch // 3, poisoned - 1, poisoned + 1} & set(range(batch))) - {poisoned})
    few = np.ascontiguousarray(feat[keep])
    pairs = [(out, orc.dlrm_fwd(few, m, k, len(keep), dtype), k)]
    if backward:
        up = uniform_bits(m * k, dtype, batch * width).reshape(batch, width)
        grad, mlp = (to_device(np.full(n, nan, dtype=np_t)) for n in (batch * m * k, batch * k))
        rw.dlrm_bwd(dev_feat, to_device(bad(up).ravel()), grad, mlp, m, k, batch, dtype)
        wgrad, wmlp = orc.dlrm_bwd(few, np.ascontiguousarray(up[keep]), m, k, len(keep), dtype)
        pairs.append((grad, wgrad, m))
        torch.cuda.synchronize()
        assert np.array_equal(mlp.cpu().numpy().view(np_t).reshape(batch, k)[keep].ravel(), np.ascontiguousarray(wmlp).ravel())
    torch.cuda.synchronize()
    for dev, ref, terms in pairs:
        got = np.ascontiguousarray(dev.cpu().numpy().view(np_t).reshape(batch, -1)[keep]).ravel()
        tol = 10 * 2.0 ** -10 if dtype == orc.F16 else max(1e-6, 2.0 * terms / 3.0 * 2.0 ** -24)
        err, inf, isnan = orc.compare_equal(dtype, got, dtype, np.ascontiguousarray(ref).ravel())
        assert not inf and not isnan and err <= tol, (err, inf, isnan)
