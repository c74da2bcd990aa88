"""The ring kernels' K loop where it can go wrong: contractions that end at every place of the ring (one K step to several rounds, each with
and without a tail), slices that switch at every place, and the tiles on three stages split and behind the input gate."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib, local_gemm
from meshslice_amd.slice_layout import pack_slices

pytestmark = pytest.mark.gpu


def _rand(g, rows, cols, scale=1.0):
    return (torch.randn(rows, cols, generator=g, device="cuda") * scale).bfloat16()


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("variant", [1, 2, 3, 4, 5, 7, 8, 14])
def test_contractions_that_end_at_every_place_of_the_ring(variant, flow):
    """fp32 sums of at most 1400 exact products against float64: their roundings, 2^-24 each, add up to well under 1e-5."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(variant)
    m, n = 200, 264
    try:
        assert lib.ms_set_variant(variant) == 0
        for S, k in [(1, k) for k in (8, 56, 64, 72, 128, 136, 192, 200, 256, 264, 320, 384, 448, 456)] + [(2, 72), (3, 64), (3, 200), (4, 136), (5, 280)]:
            if flow == "os":
                A, B = [_rand(g, m, k) for _ in range(S)], [_rand(g, k, n) for _ in range(S)]
                got, want = [ms.gemm_os(A, B, out_dtype=torch.float32)], [sum(a.double() @ b.double() for a, b in zip(A, B))]
            elif flow == "ls":
                A, W = _rand(g, m, k), [_rand(g, n, k) for _ in range(S)]
                got, want = ms.gemm_ls(A, W), [A.double() @ w.double().t() for w in W]
            else:
                X, W = [_rand(g, k, m) for _ in range(S)], _rand(g, k, n)
                got, want = ms.gemm_rs(X, W), [x.double().t() @ W.double() for x in X]
            assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == variant
            for y, w in zip(got, want, strict=True):
                assert float((y.double() - w).norm() / w.norm()) <= 1e-5, (S, k)
    finally:
        lib.ms_set_variant(0)


@pytest.mark.parametrize("splits", [2, 3, 8])
@pytest.mark.parametrize("m,n,k,S", [(128, 192, 512, 1), (300, 400, 328, 4), (520, 1000, 1544, 2)])
def test_the_128x192_tile_splits_its_contraction(m, n, k, S, splits):
    """Parts that end inside a slice, rows and columns that end inside a tile: the unsplit sums to their roundings, the same bits
    from run to run, bf16 as one rounding of them, and the arrival counters left clear."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(m + splits)
    A, B = [_rand(g, m, k) for _ in range(S)], [_rand(g, k, n) for _ in range(S)]
    want = sum(a.double() @ b.double() for a, b in zip(A, B))
    try:
        assert lib.ms_set_variant(4 + 100 * splits) == 0
        got = ms.gemm_os(A, B, out_dtype=torch.float32)
        assert (lib.ms_query(_lib.MS_QUERY_LAST_VARIANT), lib.ms_query(_lib.MS_QUERY_LAST_SPLITS)) == (4, splits)
        assert torch.equal(ms.gemm_os(A, B, out_dtype=torch.float32), got)
        assert torch.equal(ms.gemm_os(A, B), got.bfloat16())
    finally:
        lib.ms_set_variant(0)
    assert float((got.double() - want).norm() / want.norm()) <= 1e-5
    torch.cuda.synchronize()
    assert int(local_gemm.workspace("cuda:0")[:4096].view(torch.int32).abs().sum()) == 0


def test_the_128x192_tile_behind_the_input_gate():
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(4)
    A, B = [_rand(g, 300, 200) for _ in range(3)], [_rand(g, 200, 400) for _ in range(3)]
    try:
        assert lib.ms_set_variant(4) == 0
        want = ms.gemm_os(A, B)
        ready = torch.ones(4, dtype=torch.int32, device="cuda")
        ready[3] = 0
        assert torch.equal(ms.gemm_os_gated(A, B, ready), want)
        assert not local_gemm.gate_timed_out(ready)
    finally:
        lib.ms_set_variant(0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S,k,m,n", [(2, 8, 8, 8), (3, 72, 136, 200), (8, 24, 300, 264), (5, 136, 520, 776), (16, 64, 257, 1544), (64, 16, 64, 136)])
def test_products_on_row_slices_in_place_have_the_bits_of_copied_slices(S, k, m, n, dtype):
    """Slices of one block to several K steps with and without a tail, rows and columns that end inside a tile, W a window of a wider
    matrix, on the library's choice and on every tile."""
    g = torch.Generator(device="cuda").manual_seed(S * k)
    A = [torch.randn(m, k, generator=g, device="cuda").to(dtype) for _ in range(S)]
    W = torch.randn(S * k, n + 16, generator=g, device="cuda").to(dtype)[:, 8:8 + n]
    B = pack_slices(W, S, 8, 0)
    lib = _lib.load()
    try:
        for variant in [0] + (list(range(1, 15)) + [204, 407] if dtype == torch.bfloat16 else [21, 22, 23, 24, 25, 224]):
            assert lib.ms_set_variant(variant) == 0
            try:
                want = ms.gemm_os(A, B)
            except ValueError:       # (a split that these sizes do not take)
                continue
            assert torch.equal(local_gemm.gemm_os_cyclic(A, W), want), variant
    finally:
        lib.ms_set_variant(0)


def test_row_slices_in_place_are_checked():
    a, w = torch.randn(16, 24, device="cuda").bfloat16(), torch.randn(48, 32, device="cuda").bfloat16()
    for bad in (lambda: local_gemm.gemm_os_cyclic([a], w), lambda: local_gemm.gemm_os_cyclic([a, a], w.t()), lambda: local_gemm.gemm_os_cyclic([a[:, :12], a[:, :12]], w[:24])):
        with pytest.raises(ValueError):
            bad()
