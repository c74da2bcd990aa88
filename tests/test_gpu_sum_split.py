"""When a sum over devices gives every device's share a workgroup of its own: not for shares so short that the exchange costs more than it gives."""
import pytest
import torch

from meshslice_amd import _lib, local_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flow,P,m,n,k,parts", [("rs", 4, 384, 3712, 736, 1), ("ls", 4, 411, 1280, 280, 1), ("rs", 2, 224, 544, 319, 1), ("ls", 2, 1069, 256, 416, 1),
                                                ("rs", 8, 128, 192, 2472, 8), ("ls", 8, 162, 1088, 5304, 8), ("rs", 2, 640, 1008, 2852, 2), ("ls", 4, 772, 128, 936, 4)])
def test_short_shares_stay_whole(flow, P, m, n, k, parts):
    """(microseconds whole and in parts: 23.0 / 29.5, 16.6 / 20.2, 11.6 / 13.1, 13.0 / 14.3; 99 / 26, 348 / 58, 42 / 28, 26 / 17)"""
    g = torch.Generator(device="cuda").manual_seed(m)
    R = lambda r, c: torch.randn(r, c, generator=g, device="cuda").bfloat16()
    X, W = (R(m, k * P), R(n, k * P)) if flow == "ls" else (R(k * P, m), R(k * P, n))
    got = (local_gemm.gemm_ls_sum if flow == "ls" else local_gemm.gemm_rs_sum)(X, W, P)
    assert _lib.load().ms_query(_lib.MS_QUERY_LAST_SPLITS) == parts
    want = X.double() @ W.double().t() if flow == "ls" else X.double().t() @ W.double()
    assert float((got.double() - want).norm() / want.norm()) <= 2.0 ** -8      # one rounding to bf16
