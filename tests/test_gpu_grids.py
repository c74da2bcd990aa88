"""Grids of any size: the workgroups' order over the XCDs and the tiles' walk leave out no tile."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 7), (9, 1), (2, 5), (19, 3), (3, 19), (5, 13), (27, 9), (17, 15), (16, 16), (1, 255), (37, 11)])
@pytest.mark.parametrize("variant", [14, 3, 4, 2, 314, 24, 28])
def test_every_tile_once(rows, cols, variant):
    """rows x cols tiles, the last ones partly filled, on outputs that begin as NaN; partial sums in a row's and a column's count, exact in
    fp32, so that the expected values are exact."""
    tile_m, tile_n = {4: (128, 192), 2: (192, 192), 24: (64, 64), 28: (32, 32)}.get(variant, (128, 128))
    dtype = torch.bfloat16 if variant % 100 < 21 else torch.float32
    m, n, k = rows * tile_m - 8, cols * tile_n - 8, 256
    lib = _lib.load()
    i, j = torch.arange(m, device="cuda") % 61 - 30, torch.arange(n, device="cuda") % 53 - 26
    A, B = torch.zeros(m, k, device="cuda"), torch.zeros(k, n, device="cuda")
    A[:, 3], A[:, 200], B[3], B[200] = i.float(), 1.0, 64.0, j.float()
    want = 64.0 * i[:, None].float() + j[None].float()
    A, B = A.to(dtype), B.to(dtype)
    out = torch.full((m, n), float("nan"), device="cuda")
    chunk = [torch.full((m, n), float("nan"), device="cuda") for _ in range(2)]
    assert lib.ms_set_variant(variant) == 0
    try:
        if variant < 100 or rows * cols * (variant // 100) <= torch.cuda.get_device_properties(0).multi_processor_count:
            ms.gemm_os([A], [B], out=out, out_dtype=torch.float32)
            assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == variant % 100 and torch.equal(out, want)
        if variant < 100:
            W = B.t().contiguous()
            ms.gemm_ls(A, [W, W], out=chunk)
            assert all(torch.equal(c, want) for c in chunk)
    finally:
        lib.ms_set_variant(0)


def test_answers_kept_for_a_grid_are_that_grids():
    """Grids that share a place in the table of kept answers (19 tiles of 128 x 128 whichever way they lie, as chunks and as one output), in
    turns and again: the first call's bits each time."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(19)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    calls = []
    for rows, cols in ((19, 1), (1, 19), (3, 7), (7, 3), (9, 13), (13, 9), (17, 13), (13, 17)):
        A, B = r(rows * 128 - 40, 96), r(96, cols * 128 - 24)
        W = B.t().contiguous()
        calls += [lambda A=A, B=B: ms.gemm_os([A], [B]), lambda A=A, W=W: ms.gemm_ls(A, [W, W], out_dtype=torch.bfloat16)[1]]
    assert lib.ms_set_variant(14) == 0
    try:
        first = [f() for f in calls]
        for f, want in list(zip(calls, first)) * 2 + list(zip(calls, first))[::-1]:
            assert torch.equal(f(), want) and float((want.float() - first[calls.index(f) // 2 * 2].float()).abs().max()) == 0.0
    finally:
        lib.ms_set_variant(0)
