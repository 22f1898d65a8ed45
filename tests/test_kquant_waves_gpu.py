"""The K-quant lane GEMV with four waves sharing the activations against the oracle, bit for bit: on both sides of the
rule's lines (row lengths, lanes, the LDS limit), with waves that have no group, a partial last group, and several groups
per wave."""
import numpy as np
import pytest

import kquant_blocks as KB
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ty,k,nr,nl", [(4, 2048, 5, 2), (4, 2048, 13001, 2), (4, 1792, 66, 4), (4, 8192, 21, 4), (5, 2048, 3, 3),
                                        (5, 3072, 70, 2), (6, 3072, 19, 1), (6, 2560, 19, 1), (6, 8192, 35, 2), (6, 2048, 9000, 4),
                                        (3, 3072, 50, 2), (3, 2048, 50, 3), (3, 2048, 50, 2), (3, 8192, 17, 4)])
def test_vl_gemv_waves_match_oracle(dev, ty, k, nr, nl):
    import oxe_amd as A
    import torch
    print(f"vl_gemv type {ty} k {k} nr {nr} nl {nl}", flush=True)
    w = KB.random_blocks(ty, nr, k, seed=1000 * ty + k + nr)
    x = np.random.default_rng(nr + k).standard_normal((nl, k)).astype(np.float32)
    yd = A.quantize_q8_K(torch.from_numpy(x).to(dev))
    got = A.vl_gemv(ty, torch.from_numpy(w).to(dev), k, yd)
    want = O.vl_gemv(ty, w, k, yd.cpu().numpy())
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
