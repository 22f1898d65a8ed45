"""The Q8_0 GEMV's row counts per workgroup and its general-length kernel against the oracle, bit for bit: on both sides of
the rules' lines (matrices of 2^19 and, of short rows, 7 * 2^17 weights; 256 and 512 workgroups; rows of 4096 at 1024, 2048 and 4096 rows;
long rows of several lanes at 1536 rows), with a partial last workgroup, row lengths whose chunks
straddle a workgroup's passes, and rows too long for the general kernel's LDS."""
import numpy as np
import pytest

import oracle as O
from test_gemv_gpu import _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,nr,nl", [(1120, 468, 3), (1120, 469, 3), (1120, 3001, 4), (96, 6001, 2), (8224, 70, 1), (15360, 40, 4),
                                     (3232, 1025, 2), (2048, 4095, 1), (2048, 8193, 2), (512, 8191, 4), (512, 16385, 1),
                                     (4096, 2047, 3), (4096, 4097, 2), (65536, 9, 1), (32768, 17, 2),
                                     (320, 2867, 1), (320, 2868, 1), (320, 1876, 4), (160, 3751, 2), (160, 3751, 3), (448, 1500, 4),
                                     (12288, 1536, 3), (12288, 1537, 3), (10240, 1537, 4), (8192, 1539, 4), (9216, 1537, 4),
                                     (4096, 1024, 1), (4096, 1025, 2), (4096, 1025, 3), (4096, 2048, 4), (4096, 2049, 2), (4096, 2051, 3),
                                     (4096, 4096, 2), (4096, 4095, 4)])
def test_gemv_rows_bitexact(dev, k, nr, nl):
    import oxe_amd as A
    import torch
    wq, wd = O.synth_q8(9, 61, O.T["OUTPUT"], nr, k)
    x = O.synth_normal(9, 61 * 64 + 41, nl * k).reshape(nl, k)
    xq, xd = O.quantize_q8_0(x)
    y_ref, isum_ref = O.gemv_q8_0(wq, wd, xq, xd, want_isum=True)
    isum = torch.empty((nl, nr, k // 32), dtype=torch.int32, device=dev)
    args = [_t(a, dev) for a in (wq, wd.view(np.int16), xq, xd.view(np.int16))]
    y = A.gemv_q8_0(*args, isum=isum)
    assert np.array_equal(isum.cpu().numpy(), isum_ref)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), y_ref.view(np.uint32))
    assert torch.equal(A.gemv_q8_0(*args).view(torch.int32), y.view(torch.int32))


@pytest.mark.parametrize("k,nr,nl", [(2048, 300, 2), (4096, 1500, 1), (1120, 3001, 3), (12288, 1537, 3), (320, 1000, 2)])
def test_gemv_runs_on_the_callers_stream(dev, k, nr, nl):
    """every route's launch is recorded by a capture of the current stream; replays give the eager bits"""
    import oxe_amd as A
    import torch
    wq, wd = O.synth_q8(9, 61, O.T["OUTPUT"], nr, k)
    xq, xd = O.quantize_q8_0(O.synth_normal(9, 61 * 64 + 41, nl * k).reshape(nl, k))
    args = [_t(a, dev) for a in (wq, wd.view(np.int16), xq, xd.view(np.int16))]
    want = A.gemv_q8_0(*args)
    y = torch.zeros_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        A.gemv_q8_0(*args, y=y)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int32), want.view(torch.int32))


def test_quantize_row_tails(dev):
    """block counts around a workgroup's 32 blocks"""
    import oxe_amd as A
    rng = np.random.default_rng(3)
    for k in (32, 1024, 1056, 31 * 32):
        x = (rng.standard_normal((3, k)) * 5).astype(np.float32)
        x[1, :32] = 0.0
        q_ref, d_ref = O.quantize_q8_0(x)
        q, d = A.quantize_q8_0(_t(x, dev))
        assert np.array_equal(q.cpu().numpy(), q_ref)
        assert np.array_equal(d.cpu().numpy().view(np.uint16), d_ref)
