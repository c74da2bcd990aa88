"""Operands whose rows lie along the contraction and are so far apart that a K step's offsets, counted for all of its rows, pass 4 GiB: the rows that the slice
does not have stay zeros (offsets that wrap around would multiply some of its rows a second time).  They run on one tile of their own; a forced other one is refused."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib, local_gemm

pytestmark = pytest.mark.gpu
PITCH = 1 << 26      # bf16: rows 128 MB apart, k-row 32 lies 4 GiB on; fp32: 256 MB, k-row 16


def _far(g, rows, cols, dtype):
    t = torch.empty(rows * PITCH, dtype=dtype, device="cuda").view(rows, PITCH)[:, :cols]
    return t.copy_(torch.randn(rows, cols, generator=g, device="cuda"))


def _limit(k):
    """k products of N(0, 1) values summed in fp32: k roundings of 2^-24 of sums below 64"""
    return k * 2.0 ** -24 * 64


@pytest.mark.parametrize("dtype,k,tile", [(torch.bfloat16, 8, 14), (torch.bfloat16, 3, 14), (torch.float32, 7, 24)])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_rows_beyond_a_slice_are_zeros(dtype, k, tile, out):
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(k)
    q = 16 // torch.empty(0, dtype=dtype).element_size()
    for m, n in ((9 * q, 14 * q), (136, 264)):
        X, W = _far(g, k, m, dtype), _far(g, k, n, dtype)
        want = X.double().t() @ W.double()
        got = ms.gemm_rs([X], W, out_dtype=out)[0]
        assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == tile
        rounded = 0 if out == torch.float32 else 2.0 ** -9 * 64
        assert float((got.double() - want).abs().max()) <= _limit(k) + rounded
        # the other operand's zeros against rows that hold an infinity
        kos = k // q * q or q
        if kos <= k:
            A, B = torch.zeros(m, kos, device="cuda", dtype=dtype), W[:kos]
            A[:, 1] = A[0, 0] = 1
            B[:2] = 0
            B[1] = 2
            B[0, 0] = float("inf")
            want = torch.full((m, n), 2.0, device="cuda")
            want[:, 0] = float("nan")      # 0 x inf in every row but the first
            want[0, 0] = float("inf")
            got = ms.gemm_os([A], [B], out_dtype=out).float()
            assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == tile
            assert torch.equal(got.nan_to_num(nan=-1.0, posinf=-2.0), want.nan_to_num(nan=-1.0, posinf=-2.0))


def test_fused_gated_and_summed():
    g = torch.Generator(device="cuda").manual_seed(3)
    A, B = torch.randn(40, 8, generator=g, device="cuda").bfloat16(), _far(g, 8, 72, torch.bfloat16)
    R = torch.randn(40, 72, generator=g, device="cuda").bfloat16()
    plain = ms.gemm_os([A, A], [B, B], out_dtype=torch.float32)
    assert float((plain.double() - 2 * (A.double() @ B.double())).abs().max()) <= _limit(16)
    assert torch.equal(ms.gemm_os([A, A], [B, B], residual=R), (plain + R.float()).bfloat16())
    assert torch.equal(ms.gemm_os([A, A], [B, B], out_dtype=torch.float32, residual=R.float()), plain + R.float())
    ready = torch.tensor([1, 1, 0], dtype=torch.int32, device="cuda")
    assert torch.equal(ms.gemm_os_gated([A, A], [B, B], ready, out_dtype=torch.float32), plain)
    W = _far(g, 8, 40, torch.bfloat16)
    got = local_gemm.gemm_rs_sum(B, W, 2)
    assert _lib.load().ms_query(_lib.MS_QUERY_LAST_VARIANT) == 15      # (that tile with the devices' sums)
    assert torch.equal(got, sum(ms.gemm_rs([B[4 * p:4 * p + 4]], W[4 * p:4 * p + 4])[0] for p in range(2)).bfloat16())


def test_other_tiles_are_refused():
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(4)
    try:
        for dtype, own, others in ((torch.bfloat16, 14, (2, 7, 12, 18, 19, 214, 200)), (torch.float32, 24, (21, 25, 28, 224))):
            X, W = _far(g, 4, 64, dtype), _far(g, 4, 64, dtype)
            want = X.double().t() @ W.double()
            for v in others:
                assert lib.ms_set_variant(v) == 0
                with pytest.raises(_lib.MeshSliceError, match="does not reach rows of more than"):
                    ms.gemm_os([torch.zeros(8, 4 if dtype == torch.float32 else 8, dtype=dtype, device="cuda")], [_far(g, 4 if dtype == torch.float32 else 8, 64, dtype)])
            assert lib.ms_set_variant(own) == 0
            assert float((ms.gemm_rs([X], W)[0].double() - want).abs().max()) <= _limit(4)
    finally:
        lib.ms_set_variant(0)
