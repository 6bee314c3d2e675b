"""Block-scaled GEMM on scales in the caller's order (no re-ordering launch) against the same problem on scales re-ordered
beforehand: the products and their order are the same, so the results must be equal bit for bit.  Sizes at the edges of the
tiles and of the pairs of stages, either side of the rule that chooses, padded and unaligned scale rows (which go through
the re-ordering launch), NaN scales, and a column-major C."""
import numpy as np
import pytest

import rocwmma_amd as rw

pytestmark = pytest.mark.gpu

# (m, n, k): 128 x 128 tiles in one round and two, 128 x 64 tiles on the ring of two (K below 4 KiB) and of four, one tile row
# more and less than filled, odd and even counts of 128-byte stages, the shortest K of the path and one below it
SHAPES = [(48, 1040, 256), (48, 1040, 128), (128, 1024, 384), (144, 2064, 640), (112, 4112, 4224), (64, 8208, 4096), (272, 4096, 4352),
          (1040, 2064, 256), (2000, 3056, 1408), (1024, 4112, 1664), (2064, 8208, 384), (128, 1024, 3968)]


@pytest.mark.parametrize("pad,shift,nan,col", [(0, 0, False, False), (4, 4, True, False), (1, 0, False, False), (0, 1, False, False), (8, 0, False, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_raw_scales_equal_packed(m, n, k, pad, shift, nan, col):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn((m, k), device="cuda", generator=gen).to(torch.float8_e4m3fn)
    b = torch.randn((n, k), device="cuda", generator=gen).to(torch.float8_e4m3fn)
    ld = k // 32 + pad

    def scales(rows):
        flat = torch.randint(118, 130, (shift + rows * ld,), generator=gen, device="cuda", dtype=torch.uint8)
        view = flat[shift:]
        if nan:
            view[(rows // 2) * ld + k // 64] = 255
        return view

    sa, sb = scales(m), scales(n)
    if col:  # the same numbers as an n x m problem with a column-major result
        call, ops, scl = (rw.ROW_MAJOR, rw.COL_MAJOR, rw.COL_MAJOR, n, m, k), (b, a), (sb, sa)
    else:
        call, ops, scl = (rw.ROW_MAJOR, rw.COL_MAJOR, rw.ROW_MAJOR, m, n, k), (a, b), (sa, sb)
    size = rw.gemm_mx_workspace_size(call[3], call[4], k)
    d, want = (torch.full((m, n), 7.0, device="cuda") for _ in range(2))
    w1, w2 = (torch.zeros(size, dtype=torch.uint8, device="cuda") for _ in range(2))
    rw.gemm_mx(rw.E4M3, *call, ops[0], scl[0], ops[1], scl[1], None, d, 1.0, 0.0, w1, ld_scale_a=ld, ld_scale_b=ld)
    rw.gemm_mx_pack_scales(*call, scl[0], scl[1], w2, ld_scale_a=ld, ld_scale_b=ld)
    rw.gemm_mx_packed(rw.E4M3, *call, ops[0], ops[1], None, want, 1.0, 0.0, w2)
    torch.cuda.synchronize()
    got, ref = d.cpu().numpy(), want.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and bool(np.isnan(ref).any()) == nan
    assert np.array_equal(got[~np.isnan(ref)].view(np.uint32), ref[~np.isnan(ref)].view(np.uint32))
