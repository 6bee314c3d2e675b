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
          (1040, 2064, 256), (2000, 3056, 1408), (1024, 4112, 1664), (2064, 8208, 384), (128, 1024, 3968),
          (96, 8208, 8192), (96, 8208, 8320), (272, 4096, 5760)]


# of SHAPES, on 256 compute units: the ones that go through the re-ordering launch even with aligned scales
REORDERED = [(48, 1040, 128), (1024, 4112, 1664), (128, 1024, 3968), (96, 8208, 8320), (272, 4096, 5760)]


def launches_of(call):
    """Kernels that `call` enqueues: the nodes of its captured graph."""
    import ctypes

    import torch

    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    nodes = ctypes.c_size_t(0)
    get = ctypes.CDLL(path).hipGraphGetNodes
    get.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    assert get(graph.raw_cuda_graph(), None, ctypes.byref(nodes)) == 0
    return nodes.value


def problem(m, n, k, pad, shift, nan, col):
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
    return call, ops, scl, ld


@pytest.mark.parametrize("pad,shift,nan,col", [(0, 0, False, False), (4, 4, True, False), (1, 0, False, False), (0, 1, False, False), (8, 0, False, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_raw_scales_equal_packed(m, n, k, pad, shift, nan, col):
    import torch

    call, ops, scl, ld = problem(m, n, k, pad, shift, nan, col)
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


@pytest.mark.parametrize("pad,shift,nan,col", [(0, 0, False, False), (4, 4, True, False), (1, 0, False, False), (8, 0, False, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_workspace_holds_the_packed_scales_afterwards(m, n, k, pad, shift, nan, col):
    """Whichever way a call reads its scales, it leaves them in the workspace as the re-ordering call does, byte for byte."""
    import torch

    call, ops, scl, ld = problem(m, n, k, pad, shift, nan, col)
    size = rw.gemm_mx_workspace_size(call[3], call[4], k)
    d, again = (torch.full((m, n), 7.0, device="cuda") for _ in range(2))
    guard = 256
    w1, w2 = (torch.full((size + guard,), 0xA5, dtype=torch.uint8, device="cuda") for _ in range(2))
    rw.gemm_mx(rw.E4M3, *call, ops[0], scl[0], ops[1], scl[1], None, d, 1.0, 0.0, w1[:size], ld_scale_a=ld, ld_scale_b=ld)
    rw.gemm_mx_pack_scales(*call, scl[0], scl[1], w2[:size], ld_scale_a=ld, ld_scale_b=ld)
    assert torch.equal(w1, w2)
    # the weights' scales stay, the tokens' are re-ordered alone, and the product runs on the workspace
    rw.gemm_mx_pack_scales(*call, scl[0], None, w1[:size], ld_scale_a=ld, ld_scale_b=ld)
    rw.gemm_mx_packed(rw.E4M3, *call, ops[0], ops[1], None, again, 1.0, 0.0, w1[:size])
    assert torch.equal(d.view(torch.int32), again.view(torch.int32))


@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 4), (1, 0), (0, 1)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_which_problems_read_raw_scales(m, n, k, pad, shift):
    """One launch on scales as they are, two with the re-ordering in front (unaligned scale rows always)."""
    import torch

    if rw.device_info()["compute_units"] != 256:
        pytest.skip("the rule goes by the compute units")
    call, ops, scl, ld = problem(m, n, k, pad, shift, False, False)
    d = torch.empty((m, n), device="cuda")
    work = torch.empty(rw.gemm_mx_workspace_size(m, n, k), dtype=torch.uint8, device="cuda")
    run = lambda: rw.gemm_mx(rw.E4M3, *call, ops[0], scl[0], ops[1], scl[1], None, d, 1.0, 0.0, work, ld_scale_a=ld, ld_scale_b=ld)
    run()
    aligned = pad % 4 == 0 and shift % 4 == 0
    assert launches_of(run) == (1 if aligned and (m, n, k) not in REORDERED else 2)
