"""The 64x64 and 64x128 tiles (ids 18 and 19) in every form that a product comes in: slices in place, several devices' pointers, completion counters, windows,
sixty-four slices, grids of any size, sums over devices beside them, and slices that arrive after the launch."""
import time

import pytest
import torch

import meshslice_amd as ms
import test_gpu_grids as grids
import test_gpu_signal as signals
import test_gpu_sum as sums
import test_gpu_whole_mesh as whole_mesh
import test_zx_gpu_gate as gate
from meshslice_amd import _lib, local_gemm
from meshslice_amd.slice_layout import pack_slices

pytestmark = pytest.mark.gpu
TILES = pytest.mark.parametrize("tile", [18, 19])


@pytest.fixture(autouse=True)
def _default_variant():
    yield
    _lib.load().ms_set_variant(0)


def _rand(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda").bfloat16()


@pytest.mark.parametrize("variant", [18, 19, 218, 318, 219, 419])
@pytest.mark.parametrize("S,k,m,n", [(2, 8, 8, 8), (3, 72, 136, 200), (8, 24, 300, 264), (5, 136, 520, 776), (16, 64, 257, 1544), (64, 16, 64, 136), (2, 1160, 72, 200), (3, 264, 40, 64)])
def test_row_slices_in_place_along_the_contraction(S, k, m, n, variant):
    """OS on W's rows where they lie: sixteen blocks of eight rows a step, K tails, W a window whose neighbours are NaN; the bits of the copied slices."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(S * k)
    A = [_rand(g, m, k) for _ in range(S)]
    wide = torch.full((S * k, n + 16), float("nan"), device="cuda", dtype=torch.bfloat16)
    W = wide[:, 8:8 + n].copy_(_rand(g, S * k, n))
    assert lib.ms_set_variant(variant) == 0
    tiles = -(-m // 64) * -(-n // (64 if variant % 100 == 18 else 128))
    step = 128 if variant % 100 == 18 else 64
    if variant > 100 and (tiles * (variant // 100) > 256 or tiles > 128 or -(-k // step) * S < variant // 100):
        with pytest.raises(ValueError):
            local_gemm.gemm_os_cyclic(A, W)
        return
    got = local_gemm.gemm_os_cyclic(A, W)
    assert (lib.ms_query(_lib.MS_QUERY_LAST_VARIANT), lib.ms_query(_lib.MS_QUERY_LAST_SPLITS)) == (variant % 100, max(1, variant // 100))
    assert torch.equal(got, ms.gemm_os(A, pack_slices(W, S, 8, 0)))
    if variant < 100:
        lib.ms_set_variant(14)
        assert torch.equal(got, local_gemm.gemm_os_cyclic(A, W))


@TILES
@pytest.mark.parametrize("S,n,m,k", [(2, 8, 8, 8), (3, 136, 72, 200), (8, 264, 300, 72), (16, 264, 257, 1544), (64, 16, 64, 136), (1, 640, 100, 264)])
def test_row_slices_in_place_as_chunks(S, n, m, k, tile):
    g = torch.Generator(device="cuda").manual_seed(S * n)
    A = _rand(g, m, k)
    wide = torch.full((S * n, k + 16), float("nan"), device="cuda", dtype=torch.bfloat16)
    W = wide[:, 8:8 + k].copy_(_rand(g, S * n, k))
    lib = _lib.load()
    assert lib.ms_set_variant(tile) == 0
    got = local_gemm.gemm_ls_cyclic(A, W, S)
    assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == tile
    lib.ms_set_variant(14)
    assert all(torch.equal(a, b) for a, b in zip(got, ms.gemm_ls(A, pack_slices(W, S, 8, 0)), strict=True))


@TILES
@pytest.mark.parametrize("flow,P,S", [("ls", 2, 3), ("ls", 4, 1), ("rs", 2, 3), ("rs", 4, 1)])
def test_several_devices_pointers(tile, flow, P, S):
    whole_mesh.test_peers_products_on_every_tile_equal_the_single_devices(tile, flow, P, S)


@TILES
@pytest.mark.parametrize("flow", ["ls", "rs"])
def test_counted_chunks(flow, tile):
    signals.test_counted_chunks_equal_the_plain_call_and_every_counter_ends_at_the_tile_count(flow, tile)


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 7), (9, 1), (2, 5), (19, 3), (3, 19), (5, 13), (27, 9), (17, 15), (16, 16), (37, 11)])
@pytest.mark.parametrize("variant", [18, 19, 218, 319])
def test_grids_of_any_size(rows, cols, variant):
    """rows x cols tiles of 64x64 (the walk's own test has 128x128 ones): every tile once."""
    lib = _lib.load()
    m, n, k = rows * 64 - 8, cols * (64 if variant % 100 == 18 else 128) - 8, 512
    i, j = torch.arange(m, device="cuda") % 61 - 30, torch.arange(n, device="cuda") % 53 - 26
    A, B = torch.zeros(m, k, device="cuda"), torch.zeros(k, n, device="cuda")
    A[:, 3], A[:, 400], B[3], B[400] = i.float(), 1.0, 64.0, j.float()
    want = 64.0 * i[:, None].float() + j[None].float()      # exact
    out = torch.full((m, n), float("nan"), device="cuda")
    assert lib.ms_set_variant(variant) == 0
    if variant < 100 or (rows * cols * (variant // 100) <= 256 and rows * cols <= 128):      # (what a split product may have)
        ms.gemm_os([A.bfloat16()], [B.bfloat16()], out=out, out_dtype=torch.float32)
        assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == variant % 100 and torch.equal(out, want)
    if variant < 100:
        grids.test_every_tile_once(rows, cols, variant)


@TILES
@pytest.mark.parametrize("flow", ["ls", "rs"])
def test_a_global_product_on_it(tile, flow):
    sums.test_a_forced_tile_runs_global_products(tile, flow)


@TILES
@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("m,n,k", [(520, 776, 1000), (264, 392, 9000)])
def test_the_order_of_the_additions(m, n, k, flow, tile):
    """Operands spread over e^+-8, so that another order than the other tiles' would show; windows of wider matrices."""
    g = torch.Generator(device="cuda").manual_seed(k)
    r = lambda a, b: (torch.randn(a, b + 24, generator=g, device="cuda") * torch.exp(4 * torch.randn(a, b + 24, generator=g, device="cuda"))).bfloat16()[:, 16:16 + b]
    a, b = {"os": ((m, k), (k, n)), "ls": ((m, k), (n, k)), "rs": ((k, m), (k, n))}[flow]
    a, b = r(*a), r(*b)
    run = {"os": lambda: ms.gemm_os([a], [b], out_dtype=torch.float32), "ls": lambda: ms.gemm_ls(a, [b])[0], "rs": lambda: ms.gemm_rs([a], b)[0]}[flow]
    lib = _lib.load()
    results = []
    for v in (14, tile):
        _lib.check(lib.ms_set_variant(v))
        results.append(run())
        assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) == v
    assert torch.equal(*results)


@TILES
@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_sixty_four_slices(flow, tile):
    g = torch.Generator(device="cuda").manual_seed(64)
    S, m, n, k = 64, 72, 72, 40
    if flow == "os":
        A, B = [_rand(g, m, k) for _ in range(S)], [_rand(g, k, n) for _ in range(S)]
        run = lambda: [ms.gemm_os(A, B, out_dtype=torch.float32)]
    elif flow == "ls":
        A, W = _rand(g, m, k), [_rand(g, n, k) for _ in range(S)]
        run = lambda: ms.gemm_ls(A, W)
    else:
        X, W = [_rand(g, k, m) for _ in range(S)], _rand(g, k, n)
        run = lambda: ms.gemm_rs(X, W)
    lib = _lib.load()
    lib.ms_set_variant(14)
    want = run()
    lib.ms_set_variant(tile)
    assert all(torch.equal(a, b) for a, b in zip(run(), want, strict=True))


@pytest.mark.parametrize("tile", [0, 18, 19])
@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_slices_that_arrive_after_the_launch(flow, tile, stream_beside):
    """The gathered operands hold zeros at the launch; a second stream fills them (OS: in order, the others last slice first) and raises each flag.  A load ahead
    of its flag would bring zeros.  Short and long slices: steps that reach into the next one while the first is under the MFMAs."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(tile + 1)
    cur = torch.cuda.current_stream()
    producer = stream_beside(cur)
    for S, m, n, k in ((4, 200, 328, 264), (6, 136, 200, 72), (2, 328, 136, 1160)):
        if flow == "os":
            own, src = None, [[_rand(g, m, k) for _ in range(S)], [_rand(g, k, n) for _ in range(S)]]
        else:
            own, src = (_rand(g, m, k), [[_rand(g, n, k) for _ in range(S)]]) if flow == "ls" else (_rand(g, k, n), [[_rand(g, k, m) for _ in range(S)]])
        dst = [[torch.zeros_like(t) for t in ts] for ts in src]
        plain = {"os": lambda o: [ms.gemm_os(*o)], "ls": lambda o: ms.gemm_ls(own, o[0]), "rs": lambda o: ms.gemm_rs(o[0], own)}[flow]
        ready = torch.zeros(S + 1, dtype=torch.int32, device="cuda")
        gated = {"os": lambda o: [ms.gemm_os_gated(*o, ready, timeout_ms=1500)], "ls": lambda o: ms.gemm_ls_gated(own, o[0], ready, timeout_ms=1500),
                 "rs": lambda o: ms.gemm_rs_gated(o[0], own, ready, timeout_ms=1500)}[flow]
        try:
            assert lib.ms_set_reserved_cus(32) == 0      # the copies need compute units beside the waiting product
            assert lib.ms_set_variant(tile) == 0
            want = plain(src)
            torch.cuda.synchronize()
            got = gated(dst)
            assert tile in (0, lib.ms_query(_lib.MS_QUERY_LAST_VARIANT))
        finally:
            lib.ms_set_reserved_cus(0)
            lib.ms_set_variant(0)
        time.sleep(0.003)                                # the product is on the device and waiting
        with torch.cuda.stream(producer):
            for s in range(S) if flow == "os" else reversed(range(S)):
                for d, t in zip(dst, src):
                    d[s].copy_(t[s])
                ms.signal_set(ready, s)
        torch.cuda.synchronize()
        assert not ms.gate_timed_out(ready)
        assert all(torch.equal(a, b) for a, b in zip(got, want, strict=True)), (S, m, n, k)


@TILES
@pytest.mark.parametrize("flow", ["ls", "rs"])
def test_every_flag_set_and_counted(tile, flow):
    gate.test_with_every_flag_set_the_gated_chunk_calls_equal_the_plain_ones(tile, torch.bfloat16, flow)


@TILES
def test_every_flag_set(tile):
    gate.test_with_every_flag_set_the_gated_call_equals_the_plain_one(tile, torch.bfloat16)
