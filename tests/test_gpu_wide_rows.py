"""Operands whose rows lie along the contraction and are so far apart that a K step's offsets, counted for all of its rows, pass 4 GiB: the rows that the slice
does not have stay zeros (offsets that wrap around would multiply some of its rows a second time)."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib

pytestmark = pytest.mark.gpu
BF16 = [(torch.bfloat16, 8, 1 << 26, v) for v in (0, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 19)]      # rows 128 MB apart: k-row 32 lies 4 GiB on
F32 = [(torch.float32, 7, 1 << 26, v) for v in (0, 21, 22, 23, 24, 25, 28)]                               # 256 MB: k-row 16


def _far(g, rows, cols, pitch, dtype):
    t = torch.empty(rows * pitch, dtype=dtype, device="cuda").view(rows, pitch)[:, :cols]
    return t.copy_(torch.randn(rows, cols, generator=g, device="cuda"))


@pytest.fixture
def forced():
    lib = _lib.load()
    yield lambda v: lib.ms_set_variant(v)
    lib.ms_set_variant(0)


@pytest.mark.parametrize("dtype,k,pitch,variant", BF16 + F32)
def test_rows_beyond_a_slice_are_zeros(dtype, k, pitch, variant, forced):
    """At most eight products of N(0, 1) values summed in fp32: eight roundings of 2^-24 of sums below 64."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(variant)
    q = 16 // torch.empty(0, dtype=dtype).element_size()
    m, n = 9 * q, 13 * q
    X, W = _far(g, k, m, pitch, dtype), _far(g, k, n, pitch, dtype)
    want = X.double().t() @ W.double()
    assert forced(variant) == 0
    got = ms.gemm_rs([X], W, out_dtype=torch.float32)[0]
    assert variant in (0, lib.ms_query(_lib.MS_QUERY_LAST_VARIANT))
    assert float((got.double() - want).abs().max()) <= 8 * 2.0 ** -24 * 64
    # the other operand's zeros against rows that hold an infinity
    kos = 8 if dtype == torch.bfloat16 else 4
    A, B = torch.zeros(m, kos, device="cuda", dtype=dtype), _far(g, kos, n, pitch, dtype)
    A[:, 1] = 1
    B[1] = 2
    B[0] = 0
    B[0, 0] = float("inf")
    A[0, 0] = 1
    got = ms.gemm_os([A], [B], out_dtype=torch.float32)
    want = torch.full((m, n), 2.0, device="cuda")
    want[:, 0] = float("nan")      # 0 x inf in every row but the first
    want[0, 0] = float("inf")
    assert torch.equal(got.nan_to_num(nan=-1.0, posinf=-2.0), want.nan_to_num(nan=-1.0, posinf=-2.0))
