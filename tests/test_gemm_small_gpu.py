"""The Q8_0 GEMM's single-wave tiles of 16 and 32 (few tokens) through the C ABI against the oracle's GEMV, bit for
bit: around the tile edges, with one stage of K and with more and fewer stages than a wave keeps in flight, and with an
output that forbids 16-byte stores."""
import numpy as np
import pytest

import oracle as O
from test_gemm_gpu import _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,nr,nt", [(128, 16, 1), (256, 17, 16), (384, 33, 17), (640, 1000, 15), (768, 31, 33), (896, 9000, 31),
                                     (1152, 12352, 33), (2048, 2050, 65), (4096, 2048, 45), (512, 12290, 64)])
def test_small_gemm_bitexact_vs_oracle(dev, k, nr, nt):
    import oxe_amd as A
    import torch
    wq, wd = O.synth_q8(13, 3, O.T["OUTPUT"], nr, k)
    x = (O.synth_normal(13, 7 * 64 + nt, nt * k).reshape(nt, k) * 3.0).astype(np.float32)
    xq, xd = O.quantize_q8_0(x)
    y_ref = O.gemv_q8_0(wq, wd, xq, xd)
    args = [_t(a, dev) for a in (wq, wd.view(np.int16), xq, xd.view(np.int16))]
    wide = torch.full((nt, nr + 5), 7.0, device=dev)   # a row stride that is no multiple of 4 for most sizes
    for y in (A.gemm_q8_0(*args), A.gemm_q8_0(*args, y=wide[:, :nr])):
        got = y.cpu().numpy()
        bad = np.nonzero(got.view(np.uint32) != y_ref.view(np.uint32)) if got.flags.c_contiguous else np.nonzero(got != y_ref)
        assert bad[0].size == 0, f"{bad[0].size} outputs differ, first (token, row) {bad[0][0]}, {bad[1][0]}"
    assert bool((wide[:, nr:] == 7.0).all())   # nothing past the rows
