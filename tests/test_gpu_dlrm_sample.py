"""DLRM samples held whole in LDS (dlrm_sample.hip): feature counts and widths at the edges of its blocks, steps and
waves per sample, against the CPU oracle; a sample of NaNs between the others must not reach them.
Tolerances as in tests/test_gpu_dlrm.py: 10 eps of float16; float32 sums of n products of values uniform in [-1, 1]: twice
n / 3 * 2^-24 (n roundings of 2^-24 of a partial sum of about sqrt(n) / 3, on either side)."""
import numpy as np
import pytest

import oracle as orc
import rocwmma_amd as rw
from util import to_device, uniform_bits

pytestmark = pytest.mark.gpu

# (batch, m, k): one block and parts of it, a block more, the last block of every waves-per-sample choice, widths of one
# piece, of an odd and an even number of pieces, ends inside a step of K, and sizes around the LDS limits
SHAPES = [(5, 1, 8), (5, 2, 16), (7, 15, 24), (5, 16, 40), (6, 17, 72), (5, 31, 128), (9, 33, 8), (5, 41, 72), (6, 48, 200),
          (5, 64, 256), (5, 65, 120), (5, 80, 128), (5, 96, 232), (5, 113, 64), (5, 128, 16), (3, 128, 256), (5, 129, 48), (5, 161, 128),
          (3, 192, 128), (5, 27, 1024), (5, 19, 2048), (3001, 13, 56), (1501, 37, 104), (6000, 9, 16)]


def run(dtype, m, k, batch, feat, up):
    import torch

    np_t, nan = (np.uint16, 0x7E00) if dtype == orc.F16 else (np.float32, np.nan)
    width = k + m * (m - 1) // 2
    out, grad, mlp = (to_device(np.full(n, nan, dtype=np_t)) for n in (batch * width, batch * m * k, batch * k))
    rw.dlrm_fwd(to_device(feat), out, m, k, batch, dtype)
    rw.dlrm_bwd(to_device(feat), to_device(up), grad, mlp, m, k, batch, dtype)
    torch.cuda.synchronize()
    back = lambda t: t.cpu().numpy().view(np_t)
    return back(out).reshape(batch, width), back(grad).reshape(batch, m * k), back(mlp).reshape(batch, k)


@pytest.mark.parametrize("dtype", [orc.F16, orc.F32])
@pytest.mark.parametrize("batch,m,k", SHAPES)
def test_samples_in_lds(dtype, batch, m, k):
    width = k + m * (m - 1) // 2
    feat = uniform_bits(m + k, dtype, batch * m * k).reshape(batch, m * k)
    up = uniform_bits(m * k, dtype, batch * width).reshape(batch, width)
    poisoned = batch // 2
    nan = 0x7E00 if dtype == orc.F16 else np.nan
    pf, pu = feat.copy(), up.copy()
    pf[poisoned] = nan
    pu[poisoned] = nan
    out, grad, mlp = run(dtype, m, k, batch, pf.ravel(), pu.ravel())
    keep = np.arange(batch) != poisoned
    feat, up = np.ascontiguousarray(feat[keep]), np.ascontiguousarray(up[keep])
    n = batch - 1
    want = orc.dlrm_fwd(feat, m, k, n, dtype)
    wgrad, wmlp = orc.dlrm_bwd(feat, up, m, k, n, dtype)
    for got, ref, terms in ((out, want, k), (grad, wgrad, m)):
        tol = 10 * 2.0 ** -10 if dtype == orc.F16 else max(1e-6, 2.0 * terms / 3.0 * 2.0 ** -24)
        err, inf, nan = orc.compare_equal(dtype, np.ascontiguousarray(got[keep]).ravel(), dtype, np.ascontiguousarray(ref).ravel())
        assert not inf and not nan and err <= tol, (err, inf, nan)
    assert np.array_equal(np.ascontiguousarray(mlp[keep]).ravel(), np.ascontiguousarray(wmlp).ravel())
