"""Where the 64-row tiles are not chosen: RS chunks of few rows, whose time goes into streaming W."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,S,tile", [(128, 4016, 778, 16, 3), (256, 4048, 642, 16, 3), (512, 3904, 889, 16, 3), (72, 5256, 9701, 3, 14), (112, 7024, 7648, 2, 14), (48, 2632, 6867, 6, 14),
                                          (192, 4216, 3414, 3, 14), (640, 1496, 1361, 16, 19), (72, 1352, 5833, 3, 18), (128, 808, 1461, 16, 18)])
def test_thin_chunks(m, n, k, S, tile):
    """(microseconds on the 64-row tile that was chosen, and here: 18.7 / 15.3, 17.5 / 15.4, 20.0 / 15.3, 82.8 / 64.4, 54.4 / 45.9, 43.1 / 40.3, 26.9 / 23.9; the last three
    stay on theirs).  Sums of k products in fp32: 1e-5 in the norm, as every fp32 output."""
    g = torch.Generator(device="cuda").manual_seed(m)
    X, W = [torch.randn(k, m // S, generator=g, device="cuda").bfloat16() for _ in range(S)], torch.randn(k, n, generator=g, device="cuda").bfloat16()
    got = ms.gemm_rs(X, W)
    assert _lib.load().ms_query(_lib.MS_QUERY_LAST_VARIANT) == tile
    for x, y in zip(X, got):
        want = x.double().t() @ W.double()
        assert float((y.double() - want).norm() / want.norm()) <= 1e-5
