"""Products on W's row slices where they lie, and device bodies that read their peers' shards in place: the bits of the copies."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib, local_gemm
from meshslice_amd import TensorParallel as tp
from meshslice_amd.mesh import Mesh, create_device_mesh
from meshslice_amd.slice_layout import pack_slices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S,n,m,k", [(2, 8, 8, 8), (3, 136, 72, 200), (8, 264, 300, 72), (5, 776, 520, 136), (16, 264, 257, 1544), (64, 16, 64, 136), (1, 640, 100, 264)])
def test_chunks_of_row_slices_in_place_have_the_bits_of_copied_slices(S, n, m, k, dtype):
    """Slices of one block to several tiles that end inside a tile, K tails, W a window of a wider matrix, on the library's choice and on
    every tile; outside the chunks nothing is read or written that the copies do not hold (the window's neighbours are NaN)."""
    g = torch.Generator(device="cuda").manual_seed(S * n)
    A = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    wide = torch.full((S * n, k + 16), float("nan"), device="cuda", dtype=dtype)
    W = wide[:, 8:8 + k]
    W.copy_(torch.randn(S * n, k, generator=g, device="cuda").to(dtype))
    slices = pack_slices(W, S, 8, 0)
    lib = _lib.load()
    try:
        for variant in [0] + (list(range(1, 15)) if dtype == torch.bfloat16 else [21, 22, 23, 24, 25, 28]):
            assert lib.ms_set_variant(variant) == 0
            got, want = local_gemm.gemm_ls_cyclic(A, W, S), ms.gemm_ls(A, slices)
            assert len(got) == S and all(torch.equal(a, b) for a, b in zip(got, want)), variant
    finally:
        lib.ms_set_variant(0)


def test_what_it_refuses_and_both_host_paths(monkeypatch):
    a, w = torch.randn(16, 24, device="cuda").bfloat16(), torch.randn(48, 24, device="cuda").bfloat16()
    native = _lib.host.gemm_ls_cyclic(a, w, 3)
    assert native is not None

    class Declines:
        def __getattr__(self, name):
            return lambda *args: None
    monkeypatch.setattr(_lib, "host", Declines())
    assert all(torch.equal(x, y) and x.dtype == torch.float32 for x, y in zip(native, local_gemm.gemm_ls_cyclic(a, w, 3)))
    for bad in (lambda: local_gemm.gemm_ls_cyclic(a, w, 5), lambda: local_gemm.gemm_ls_cyclic(a, w, 0), lambda: local_gemm.gemm_ls_cyclic(a, w[:, :16], 2),
                lambda: local_gemm.gemm_ls_cyclic(a, w[:24], 2), lambda: local_gemm.gemm_ls_cyclic(a, w.float(), 2)):
        with pytest.raises(ValueError):
            bad()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("algorithm,B", [("meshflow", 8), ("meshflow", 4), ("collective", 8), ("wang", 8)])
def test_device_bodies_read_shards_of_one_matrix_in_place(algorithm, B, flow, dtype, monkeypatch):
    """The shards as one matrix, as a window of one at an offset that the kernels cannot address, and each device's shard as a tensor of its
    own: the same bits."""
    if B == 4 and dtype == torch.bfloat16:
        B = 16
    builder = tp.SPMD(Mesh(create_device_mesh((2, 4)), ("row", "col")), algorithm, B)
    f = {"os": builder.OS, "ls": builder.LS, "rs": builder.RS}[flow](2)
    m, n, k = (512, 256, 72) if flow == "rs" else (72, 512, 256) if flow == "ls" else (72, 256, 512)
    g = torch.Generator(device="cuda").manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    X, W = (r(k, m) if flow == "rs" else r(m, k)), (r(n, k) if flow == "ls" else r(k, n))

    def odd(t):
        buf = torch.empty(t.shape[0], t.shape[1] + 9, dtype=dtype, device="cuda")
        return buf[:, 1:1 + t.shape[1]].copy_(t)
    flat = lambda y: list(y) if isinstance(y, list) else [y]
    for i, j in ((0, 0), (1, 2)):
        got = flat(f.device(i, j)(X, W))
        grids = [[[s.clone() for s in row] for row in tp._shards(t, 2, 4)] for t in (X, W)]
        for want in (flat(f.device(i, j)(odd(X), odd(W))), flat(f.body(*grids, i, j, 2, 4, f.K, f.B))):
            assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


def test_expanded_operands_are_gathered_as_before():
    """Rows at stride 0 cannot be read in place."""
    f = tp.SPMD(Mesh(create_device_mesh((2, 2)), ("row", "col")), "collective", 8).OS(1)
    X, W = (torch.randn(1, 64, device="cuda").bfloat16().expand(64, 64) for _ in range(2))
    want = f(X.contiguous(), W.contiguous())
    assert torch.equal(f(X, W), want) and torch.equal(f.device(1, 0)(X, W), want[32:, :32])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("flow,algorithm,device", [("os", "meshflow", False), ("os", "collective", False), ("os", "collective", True), ("ls", "collective", True),
                                                   ("ls", "meshflow", True), ("rs", "collective", True)])
def test_contiguous_operands_at_an_odd_base_are_copied(flow, algorithm, device, dtype):
    """Whole rows of a flat buffer from its second element on: every pitch fits, the base does not."""
    g = torch.Generator(device="cuda").manual_seed(6)

    def odd(r, c, at=1):
        return torch.randn(r * c + at, generator=g, device="cuda").to(dtype)[at:].view(r, c)
    # the operand that is gathered lies at the odd base; a device's own shard has to be aligned
    m, n, k = 64, 96, 128
    X, W = {"os": (odd(m, k), odd(k, n)), "ls": (odd(m, k, 0), odd(n, k)), "rs": (odd(k, m), odd(k, n, 0))}[flow]
    f = getattr(tp.SPMD(Mesh(create_device_mesh((2, 1) if flow == "ls" else (1, 1) if flow == "os" else (1, 2)), ("row", "col")), algorithm, 8), flow.upper())(2)
    f = f.device(0, 0) if device else f
    want = f(X.clone(), W.clone())
    got = f(X, W)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("flow,algorithm", [("os", "meshflow"), ("rs", "meshflow"), ("os", "collective"), ("rs", "collective"), ("os", "meshflow_overlap")])
def test_windows_slid_over_a_buffer(flow, algorithm, dtype):
    """Rows closer together than they are long, farther apart than a shard's: every shard is a matrix, the whole is none."""
    g = torch.Generator(device="cuda").manual_seed(8)
    m, n, k = 64, 64, 256
    r, c = (k, m) if flow == "rs" else (m, k)
    step = c // 2
    X = torch.randn(r * step + c, generator=g, device="cuda").to(dtype).as_strided((r, c), (step, 1))
    W = torch.randn(k, n, generator=g, device="cuda").to(dtype)
    f = getattr(tp.SPMD(Mesh(create_device_mesh((1, 4)), ("row", "col")), algorithm, 8), flow.upper())(2).device(0, 1)
    got, want = f(X, W), f(X.contiguous(), W)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
