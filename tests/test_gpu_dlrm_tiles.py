"""DLRM samples that do not fit the LDS, float16 forward in tiles of 128 x 128, backward in tiles of 128 or 256 rows and columns: feature counts and widths at
the edges of its tiles, stages and 64-row strips, the last rows of the packed triangle at the end of the tensor, and both
tile sizes, against the CPU oracle; a sample of NaNs between the others must not reach them.
Tolerance as in tests/test_gpu_dlrm.py: 10 eps of float16."""
import numpy as np
import pytest

import oracle as orc
import rocwmma_amd as rw
from util import to_device, uniform_bits

pytestmark = pytest.mark.gpu

# (batch, m, k): few rows too wide for the LDS (one stage; the packed triangle shorter than a piece of it), strips and tiles
# with one row more and less, widths of one piece, around 128 and 256; batches that fill the device with either tile
SHAPES = [(3, 1, 81920), (3, 2, 65544), (3, 3, 40960), (2, 7, 20480), (2, 64, 2048), (2, 65, 2056), (3, 193, 8), (3, 255, 120),
          (3, 256, 128), (2, 257, 136), (2, 319, 256), (2, 320, 264), (2, 321, 248), (1, 449, 512), (260, 193, 72), (33, 129, 1024),
          (65, 250, 1000)]


@pytest.mark.parametrize("batch,m,k", SHAPES)
def test_tiles(batch, m, k):
    import torch

    width = k + m * (m - 1) // 2
    feat = uniform_bits(m + k, orc.F16, batch * m * k).reshape(batch, m * k)
    up = uniform_bits(m * k, orc.F16, batch * width).reshape(batch, width)
    poisoned = batch // 2 if batch > 1 else -1
    pf, pu = feat.copy(), up.copy()
    if poisoned >= 0:
        pf[poisoned] = 0x7E00
        pu[poisoned] = 0x7E00
    grad, mlp = (to_device(np.full(n, 0x7E00, dtype=np.uint16)) for n in (batch * m * k, batch * k))
    rw.dlrm_bwd(to_device(pf.ravel()), to_device(pu.ravel()), grad, mlp, m, k, batch, rw.F16)
    out = to_device(np.full(batch * width, 0x7E00, dtype=np.uint16))
    rw.dlrm_fwd(to_device(pf.ravel()), out, m, k, batch, rw.F16)
    torch.cuda.synchronize()
    # the oracle is slow at the full batches: the first, the last and the poisoned sample's neighbours
    keep = sorted({0, 1, batch - 1, max(poisoned - 1, 0), min(poisoned + 1, batch - 1)} & set(range(batch)) - {poisoned})
    wgrad, wmlp = orc.dlrm_bwd(np.ascontiguousarray(feat[keep]), np.ascontiguousarray(up[keep]), m, k, len(keep), orc.F16)
    want = orc.dlrm_fwd(np.ascontiguousarray(feat[keep]), m, k, len(keep), orc.F16)
    for dev, ref in ((grad, wgrad), (out, want)):
        got = np.ascontiguousarray(dev.cpu().numpy().view(np.uint16).reshape(batch, -1)[keep]).ravel()
        err, inf, nan = orc.compare_equal(orc.F16, got, orc.F16, np.ascontiguousarray(ref).ravel())
        assert not inf and not nan and err <= 10 * 2.0 ** -10, (err, inf, nan)
    assert np.array_equal(mlp.cpu().numpy().view(np.uint16).reshape(batch, k)[keep].ravel(), np.ascontiguousarray(wmlp).ravel())
