"""Several devices' partial sums added up inside the product (gemm_ls_sum, gemm_rs_sum) against their fp32 chunks reduced in memory."""
import ctypes

import pytest
import torch

from meshslice_amd import TensorParallel as TP, _lib, local_gemm, slice_layout
from meshslice_amd.mesh import Mesh, create_device_mesh

pytestmark = pytest.mark.gpu


def _operands(flow, m, n, k, pad=0):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    shapes = ((m, k), (n, k)) if flow == "ls" else ((k, m), (k, n))
    return [torch.randn(r, c + pad, generator=g, device="cuda").bfloat16()[:, pad // 2:pad // 2 + c] for r, c in shapes]


def _in_chunks(flow, X, W, P):
    """The same from one fp32 chunk per device: the layout kernels add them up in device order and round once."""
    if flow == "ls":
        k = X.shape[1] // P
        chunks = [local_gemm.gemm_ls(X[:, p * k:(p + 1) * k], [W[:, p * k:(p + 1) * k]]) for p in range(P)]
    else:
        k = X.shape[0] // P
        chunks = [local_gemm.gemm_rs([X[p * k:(p + 1) * k]], W[p * k:(p + 1) * k]) for p in range(P)]
    return slice_layout.unpack_chunks(chunks, 8, 1, out_dtype=torch.bfloat16)


@pytest.mark.parametrize("flow", ["ls", "rs"])
@pytest.mark.parametrize("P", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("m,n,k", [(8, 8, 8), (136, 200, 64), (384, 384, 72), (520, 776, 200), (1544, 2056, 456)])
def test_sums_inside_the_product_have_the_bits_of_reduced_chunks(m, n, k, P, flow):
    """Rows and columns that end inside a tile, devices' shares of one K step to several with and without a tail, few tiles
    (one workgroup per device and tile) and many; on the library's tile and on each that carries the sum; views at wider pitches."""
    X, W = _operands(flow, m, n, k * P, pad=16)
    f = local_gemm.gemm_ls_sum if flow == "ls" else local_gemm.gemm_rs_sum
    want = _in_chunks(flow, X, W, P)
    dense = X.double() @ W.double().t() if flow == "ls" else X.double().t() @ W.double()
    lib = _lib.load()
    try:
        for variant, kernel in ((0, None), (2, 17), (4, 16), (14, 15)):
            assert lib.ms_set_variant(variant) == 0
            got = f(X, W, P)
            assert P == 1 or kernel in (None, lib.ms_query(_lib.MS_QUERY_LAST_VARIANT))
            assert torch.equal(got, want), variant
    finally:
        lib.ms_set_variant(0)
    assert float((want.double() - dense).norm() / dense.norm()) <= 2.0 ** -8      # one rounding to bf16
    torch.cuda.synchronize()
    assert int(local_gemm.workspace("cuda:0")[:4096].view(torch.int32).abs().sum()) == 0


@pytest.mark.parametrize("flow", ["ls", "rs"])
@pytest.mark.parametrize("algorithm", ["meshflow", "collective"])
@pytest.mark.parametrize("R,C,K,u,v,w", [(4, 2, 4, 3, 2, 1), (2, 4, 8, 5, 1, 2), (1, 2, 2, 7, 3, 1), (3, 2, 3, 1, 2, 3)])
def test_global_products_have_the_same_bits_through_chunks(R, C, K, u, v, w, algorithm, flow, monkeypatch):
    q = R * C * K * 8
    m, n, k = (R * u, q * v, R * C * 8 * w) if flow == "ls" else (q * v, R * C * 8 * u, R * C * 8 * w)
    X, W = _operands(flow, m, n, k)
    f = getattr(TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), algorithm), flow.upper())(K)
    got = f(X, W)
    monkeypatch.setattr(TP, "_sums_on_chip", lambda *a: False)
    assert torch.equal(got, f(X, W))


@pytest.mark.parametrize("algorithm", ["meshflow", "collective"])
@pytest.mark.parametrize("flow,P,K,m,n,k,in_registers", [
    ("rs", 16, 2, 256, 640, 6464, False), ("ls", 16, 4, 512, 512, 2816, False), ("rs", 5, 4, 160, 320, 6080, False),      # tiles that leave the device idle, too many devices to split over
    ("rs", 4, 1, 1024, 4096, 16384, False), ("rs", 4, 2, 1024, 4096, 2048, True), ("ls", 16, 2, 512, 512, 640, True), ("ls", 2, 2, 512, 512, 8192, True)])
def test_sums_are_carried_in_registers_where_that_is_the_cheaper_way(flow, P, K, m, n, k, in_registers, algorithm, monkeypatch):
    """Either way has the other's bits; both host paths make the same choice."""
    if algorithm == "meshflow" and K == 1:
        K = 2
    X, W = _operands(flow, m, n, k * P)
    f = getattr(TP.SPMD(Mesh(create_device_mesh((1, P) if flow == "ls" else (P, 1)), ("row", "col")), algorithm), flow.upper())(K)
    lib, S = _lib.load(), K if algorithm == "meshflow" else 1
    got = f(X, W)
    assert (lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) in (15, 16, 17)) == in_registers
    assert local_gemm.prefers_sum(flow, P, S, m, n, k) == bool(lib.ms_prefers_sum(int(flow == "rs"), P, S, m, n, k)) == in_registers
    monkeypatch.setattr(local_gemm, "prefers_sum", lambda *a: not in_registers)
    assert torch.equal(got, f(X, W))
    assert (lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) in (15, 16, 17)) != in_registers


@pytest.mark.parametrize("flow", ["ls", "rs"])
@pytest.mark.parametrize("variant", range(1, 15))
def test_a_forced_tile_runs_global_products(variant, flow):
    """In registers on the tiles that carry the sum, else in chunks: the same bits; and a split count that is forced on output-stationary
    products leaves the sums to the library's choice."""
    X, W = _operands(flow, 528, 784, 2 * 200)
    f = getattr(TP.SPMD(Mesh(create_device_mesh((1, 2) if flow == "ls" else (2, 1)), ("row", "col")), "collective"), flow.upper())(1)
    g = local_gemm.gemm_ls_sum if flow == "ls" else local_gemm.gemm_rs_sum
    want, lib = f(X, W), _lib.load()
    try:
        assert lib.ms_set_variant(variant) == 0
        got, used = f(X, W), lib.ms_query(_lib.MS_QUERY_LAST_VARIANT)
        assert lib.ms_set_variant(300 + (variant if variant not in (2, 4, 14) else 0)) == 0
        assert torch.equal(g(X, W, 2), want)
    finally:
        lib.ms_set_variant(0)
    assert torch.equal(got, want) and used == {2: 17, 4: 16, 14: 15}.get(variant, variant)


def test_sums_check_their_arguments():
    x, w = torch.randn(16, 64, device="cuda").bfloat16(), torch.randn(24, 64, device="cuda").bfloat16()
    for bad in (lambda: local_gemm.gemm_ls_sum(x, w, 3), lambda: local_gemm.gemm_ls_sum(x, w.t().contiguous(), 2),
                lambda: local_gemm.gemm_rs_sum(x, w, 2), lambda: local_gemm.gemm_ls_sum(x, w, 16)):      # (windows of four elements are not 16 bytes)
        with pytest.raises(ValueError):
            bad()
    with pytest.raises(_lib.MeshSliceError):
        local_gemm.gemm_ls_sum(x.float(), w.float(), 2)
    lib = _lib.load()
    for odd in ((0, 1, 1, 512, 512, 65536), (1, 64, 2, 512, 512, 65536), (0, 4, 3, 512, 512, 65536), (1, 4, 1, 0, 512, 65536), (0, 4, 1, 512, 512, -1)):
        assert lib.ms_prefers_sum(*odd) == 1
    assert lib.ms_gemm_ls_sum(None, 64, None, 64, 2, 16, 24, 32, None, 24, 1, 1, None, 0, ctypes.c_void_p(0)) == _lib.MS_ERR_ARG
    assert lib.ms_gemm_rs_sum(None, 64, None, 64, 65, 16, 24, 32, None, 24, 1, 1, None, 0, ctypes.c_void_p(0)) == _lib.MS_ERR_ARG


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R,C,K,u,v,w", [(4, 2, 4, 3, 2, 1), (2, 4, 8, 5, 1, 2), (1, 2, 2, 7, 3, 1)])
def test_global_output_stationary_products_have_the_bits_of_copied_slices(R, C, K, u, v, w, dtype):
    g = torch.Generator(device="cuda").manual_seed(u)
    m, n, k = R * u, R * C * 8 * v, R * C * K * 8 * w
    X, W = torch.randn(m, k, generator=g, device="cuda").to(dtype), torch.randn(k, n, generator=g, device="cuda").to(dtype)
    f = TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), "meshflow").OS(K)
    assert torch.equal(f(X, W), f._whole_mesh(X, W, K, 8))
    f = TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), "collective").OS(K)
    assert torch.equal(f(X, W), f._whole_mesh(X, W, 1, 1))
