"""Global products of an emulated mesh in one launch per dataflow step against the same products device by device."""
import ctypes

import pytest
import torch

from meshslice_amd import TensorParallel as TP, _lib, local_gemm
from meshslice_amd.mesh import Mesh, create_device_mesh

pytestmark = pytest.mark.gpu

# mesh, K, B, units of (rows, columns, contraction) in the smallest extents that divide
CASES = [(4, 2, 4, 8, 3, 2, 1), (2, 4, 8, 8, 5, 1, 2), (1, 2, 2, 8, 7, 3, 1), (3, 2, 3, 8, 1, 2, 3), (2, 2, 2, 2, 9, 4, 8)]


def _operands(flow, R, C, K, B, u, v, w, dtype):
    g = torch.Generator(device="cuda").manual_seed(u * 100 + v * 10 + w)
    q, edge = R * C * K * B, R * C * 8
    m, n, k = {"os": (R * u, edge * v, q * w), "ls": (R * u, q * v, edge * w), "rs": (q * v, edge * u, R * 5 * w)}[flow]
    x, y = {"os": ((m, k), (k, n)), "ls": ((m, k), (n, k)), "rs": ((k, m), (k, n))}[flow]
    rnd = lambda s: torch.randn(s, generator=g, device="cuda").to(dtype)
    return rnd(x), rnd(y)


def _dense(flow, X, W):
    X, W = X.double().cpu(), W.double().cpu()
    return X @ W if flow == "os" else X @ W.t() if flow == "ls" else X.t() @ W


@pytest.mark.parametrize("algorithm", ["meshflow", "collective"])
@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R,C,K,B,u,v,w", CASES)
def test_whole_mesh_products_equal_the_devices_products(R, C, K, B, u, v, w, dtype, flow, algorithm, monkeypatch):
    """Both ways add the same fp32 products, OS perhaps in another order: each is one rounding (2^-9 of an element, bf16) or
    the 1e-5 of the fp32 path from the float64 product.  Operands that are windows of wider matrices, at row pitches the
    kernels can and cannot address in place, give the same bits."""
    X, W = _operands(flow, R, C, K, B, u, v, w, dtype)
    f = getattr(TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), algorithm, B), flow.upper())(K)
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-5
    got = f(X, W)
    for pad in (8, 3):
        Xp = torch.zeros(X.shape[0], X.shape[1] + pad, dtype=dtype, device="cuda")[:, pad:].copy_(X)
        Wp = torch.zeros(W.shape[0], W.shape[1] + pad, dtype=dtype, device="cuda")[:, pad:].copy_(W)
        assert torch.equal(f(Xp, Wp), got)
    monkeypatch.setattr(TP, "_fits_whole_mesh", lambda *a: False)
    each = f(X, W)
    want = _dense(flow, X, W)
    for y in (got, each):
        assert y.dtype == dtype and y.is_contiguous() and tuple(y.shape) == tuple(want.shape)
        assert float((y.double().cpu() - want).norm() / want.norm()) <= tol


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_a_mesh_whose_devices_would_be_refused_is_refused(flow):
    """Four columns of the product (LS: of the contraction) per device: not a multiple of the kernels' eight bf16 elements."""
    mesh = Mesh(create_device_mesh((1, 4)), ("row", "col"))
    rnd = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    X, W = {"os": (rnd(64, 64), rnd(64, 16)), "ls": (rnd(64, 16), rnd(64, 16)), "rs": (rnd(64, 64), rnd(64, 16))}[flow]
    with pytest.raises(ValueError):
        getattr(TP.SPMD(mesh, "meshflow"), flow.upper())(2)(X, W)


def test_peers_products_check_their_tables():
    a, w = torch.randn(16, 32, device="cuda"), torch.randn(24, 32, device="cuda")
    got = local_gemm.gemm_ls_peers([a, 2 * a], [[w, w], [w, w]])
    assert len(got) == 2 and torch.equal(got[0][1], got[0][0]) and torch.equal(got[1][0], 2 * got[0][0])
    with pytest.raises(ValueError):
        local_gemm.gemm_ls_peers([a, a], [[w, w], [w]])
    with pytest.raises(ValueError):
        local_gemm.gemm_rs_peers([[w.t().contiguous()] * 33] * 2, [w.t().contiguous()] * 2)        # 66 chunks
    lib = _lib.load()
    assert lib.ms_gemm_ls_peers(None, 32, None, 32, 2, 2, 16, 24, 32, None, 24, 0, 0, ctypes.c_void_p(0)) == _lib.MS_ERR_ARG


@pytest.mark.parametrize("flow,P,S", [("ls", 2, 3), ("ls", 4, 1), ("rs", 2, 3), ("rs", 4, 1)])
@pytest.mark.parametrize("variant", list(range(15)) + [21, 22, 23, 24, 25])
def test_peers_products_on_every_tile_equal_the_single_devices(variant, flow, P, S):
    """Every kernel takes both of its operands' pointers by chunk here.  Several tiles each way on the largest shapes
    (384x192, 256x384), ragged in all extents, a contraction of several stages with a tail; distinct shards and slices,
    views at pitches wider than their rows.  The same tile gives the same bits for one device's call (ms_gemm_ls_ex /
    ms_gemm_rs_ex), in both output types, and float64 agrees."""
    dtype = torch.float32 if variant >= 21 else torch.bfloat16
    m, n, k = 520, 776, 456 if dtype == torch.bfloat16 else 132
    g = torch.Generator(device="cuda").manual_seed(variant)
    wide = lambda r, c: torch.randn(r, c + 16, generator=g, device="cuda").to(dtype)[:, 8:8 + c]
    if flow == "ls":
        own, cut = [wide(m, k) for _ in range(P)], [[wide(n, k) for _ in range(S)] for _ in range(P)]
        single = lambda p, dt: local_gemm.gemm_ls(own[p], cut[p], out_dtype=dt)
        want = lambda p, s: own[p].double() @ cut[p][s].double().t()
    else:
        own, cut = [wide(k, n) for _ in range(P)], [[wide(k, m) for _ in range(S)] for _ in range(P)]
        single = lambda p, dt: local_gemm.gemm_rs(cut[p], own[p], out_dtype=dt)
        want = lambda p, s: cut[p][s].double().t() @ own[p].double()
    lib = _lib.load()
    bf16 = torch.empty(P * S, m, n, dtype=torch.bfloat16, device="cuda")
    table = lambda ts: _lib.ptr_array([t.data_ptr() for t in ts])[0]
    flat = [t for peer in cut for t in peer]
    try:
        assert lib.ms_set_variant(variant) == 0
        got = local_gemm.gemm_ls_peers(own, cut) if flow == "ls" else local_gemm.gemm_rs_peers(cut, own)
        used = lib.ms_query(_lib.MS_QUERY_LAST_VARIANT)
        first, second = (own, flat) if flow == "ls" else (flat, own)
        _lib.check((lib.ms_gemm_ls_peers if flow == "ls" else lib.ms_gemm_rs_peers)(
            table(first), first[0].stride(0), table(second), second[0].stride(0), P, S, m, n, k, table(bf16.unbind(0)), n,
            _lib.MS_DTYPE_F32 if dtype == torch.float32 else _lib.MS_DTYPE_BF16, _lib.MS_DTYPE_BF16, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        for p in range(P):
            each = single(p, torch.float32)
            for s in range(S):
                assert torch.equal(got[p][s], each[s])
                assert torch.equal(bf16[p * S + s], each[s].to(torch.bfloat16))
                ref = want(p, s)
                # fp32 accumulation of exact products (bf16) or the fp32 path's 1e-5
                assert float((got[p][s].double() - ref).norm() / ref.norm()) <= 1e-5
    finally:
        lib.ms_set_variant(0)
    assert variant in (0, used)


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_a_product_that_fits_memory_only_line_by_line_still_runs(flow, monkeypatch):
    """An allowance below what the partial chunks (LS, RS: 512 MiB) or the slices of all of X (OS: 128 MiB) take on the whole
    mesh; a mesh line's (32 MiB, 16 MiB), the output's parts and the output fit it.  The bodies have run device by device then."""
    monkeypatch.setattr(TP, "_sums_on_chip", lambda *a: False)      # (sums in registers need no chunks)
    R, C, K = (8, 1, 2) if flow == "os" else (16, 2, 2) if flow == "ls" else (2, 16, 2)
    m, n, k, allowance = (65536, 64, 1024, 64) if flow == "os" else (8192, 8192, 256, 420)
    a, b = {"os": ((m, k), (k, n)), "ls": ((m, k), (n, k)), "rs": ((k, n), (k, m))}[flow]
    f = getattr(TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), "meshflow"), flow.upper())(K)
    X, W = torch.randn(a, device="cuda").bfloat16(), torch.randn(b, device="cuda").bfloat16()
    want = f(X, W)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    held = []
    try:
        # what earlier work left free inside the allocator's segments counts as taken
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(10000):
                held.append(torch.empty(32 << 20, dtype=torch.uint8, device="cuda"))
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (allowance << 20)) / total)
        with pytest.raises(torch.OutOfMemoryError):
            f._whole_mesh(X, W, K, 8)
        sharded = []
        monkeypatch.setattr(TP, "_shards", lambda *a, shards=TP._shards: sharded.append(1) or shards(*a))
        got = f(X, W)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert sharded      # (cut for the devices' own bodies)
    assert torch.equal(got, want) if flow != "os" else float((got.double() - want.double()).norm() / want.double().norm()) <= 2.0 ** -8


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_the_calls_that_need_no_chunks_fall_back_too(flow, monkeypatch):
    """Where a product in one launch finds no memory for its slices, workspace or output the devices' bodies run."""
    f = getattr(TP.SPMD(Mesh(create_device_mesh((2, 2)), ("row", "col")), "meshflow"), flow.upper())(2)
    X, W = _operands(flow, 2, 2, 2, 8, 3, 1, 1, torch.bfloat16)
    want = f(X, W)
    name = {"os": "gemm_os_cyclic", "ls": "gemm_ls_sum", "rs": "gemm_rs_sum"}[flow]
    refused, call = [], getattr(local_gemm, name)

    def once(*a):
        if refused:
            return call(*a)
        refused.append(1)
        raise torch.OutOfMemoryError("no memory")
    monkeypatch.setattr(local_gemm, name, once)
    got = f(X, W)
    assert refused and float((got.double() - want.double()).norm() / want.double().norm()) <= 2.0 ** -8
