"""The fp32 kernel for small outputs (32x32 tiles, the contraction shared out over a workgroup's four waves, id 28)."""
import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import _lib, local_gemm
from meshslice_amd.slice_layout import pack_slices

pytestmark = pytest.mark.gpu
WAVES = 28


@pytest.fixture
def forced():
    lib = _lib.load()
    assert lib.ms_set_variant(WAVES) == 0
    yield lib
    lib.ms_set_variant(0)


def _operands(flow, m, n, k, S):
    """Windows of wider matrices; (call, float64 results)."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    r = lambda rows, cols: torch.randn(rows, cols + 8, generator=g, device="cuda")[:, 4:4 + cols]
    if flow == "os":
        A, B = [r(m, k) for _ in range(S)], [r(k, n) for _ in range(S)]
        return (lambda **kw: [ms.gemm_os(A, B, **kw)]), [sum(a.double() @ b.double() for a, b in zip(A, B))]
    if flow == "ls":
        A, W = r(m, k), [r(n, k) for _ in range(S)]
        return (lambda **kw: ms.gemm_ls(A, W, **kw)), [A.double() @ w.double().t() for w in W]
    X, W = [r(k, m) for _ in range(S)], r(k, n)
    return (lambda **kw: ms.gemm_rs(X, W, **kw)), [x.double().t() @ W.double() for x in X]


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("m,n,k,S", [(4, 4, 4, 1), (32, 32, 32, 1), (36, 40, 28, 1), (64, 64, 128, 2), (100, 132, 260, 3), (512, 512, 256, 4), (8, 2056, 36, 5),
                                     (1000, 72, 4100, 1), (36, 8, 516, 7), (2048, 1024, 64, 2)])
def test_against_float64(forced, m, n, k, S, flow):
    """Fewer K steps than waves to hundreds, tails, waves that begin inside a slice or a later one, rows and columns that end inside a tile,
    one tile and several rounds of them.  fp32 sums in blocks of 128 k stay within 3e-7 of float64 (1e-5 is asked of the fp32
    path); the same bits from run to run, and bf16 output is one rounding of them."""
    f, want = _operands(flow, m, n, k, S)
    got = f()
    assert forced.ms_query(_lib.MS_QUERY_LAST_VARIANT) == WAVES
    for y, w in zip(got, want, strict=True):
        assert float((y.double() - w).norm() / w.norm()) <= 1e-6
    assert all(torch.equal(a, b) for a, b in zip(got, f()))
    if n % 8 == 0:
        assert all(torch.equal(a.bfloat16(), b) for a, b in zip(got, f(out_dtype=torch.bfloat16)))


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_gated_and_counted(forced, flow):
    g = torch.Generator(device="cuda").manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    ready = torch.ones(4, dtype=torch.int32, device="cuda")
    ready[3] = 0
    if flow == "os":
        A, B = [r(100, 72) for _ in range(3)], [r(72, 132) for _ in range(3)]
        assert torch.equal(ms.gemm_os_gated(A, B, ready), ms.gemm_os(A, B))
    else:
        own, cut = (r(100, 72), [r(132, 72) for _ in range(3)]) if flow == "ls" else (r(72, 132), [r(72, 100) for _ in range(3)])
        done = torch.zeros(3, dtype=torch.int32, device="cuda")
        if flow == "ls":
            want, (got, tiles) = ms.gemm_ls(own, cut), ms.gemm_ls_gated(own, cut, ready, chunk_done=done)
        else:
            want, (got, tiles) = ms.gemm_rs(cut, own), ms.gemm_rs_gated(cut, own, ready, chunk_done=done)
        assert tiles == 4 * 5 and done.tolist() == [20, 20, 20]
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert forced.ms_query(_lib.MS_QUERY_LAST_VARIANT) == WAVES and not local_gemm.gate_timed_out(ready)


@pytest.mark.parametrize("flow", ["ls", "rs"])
def test_several_devices_and_slices_in_place(forced, flow):
    g = torch.Generator(device="cuda").manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    if flow == "ls":
        own, cut = [r(40, 68) for _ in range(2)], [[r(36, 68) for _ in range(3)] for _ in range(2)]
        got, want = local_gemm.gemm_ls_peers(own, cut), [ms.gemm_ls(o, c) for o, c in zip(own, cut)]
    else:
        own, cut = [r(68, 40) for _ in range(2)], [[r(68, 36) for _ in range(3)] for _ in range(2)]
        got, want = local_gemm.gemm_rs_peers(cut, own), [ms.gemm_rs(c, o) for o, c in zip(own, cut)]
    assert all(torch.equal(a, b) for p, q in zip(got, want) for a, b in zip(p, q))
    A, W = [r(40, 24) for _ in range(5)], r(120, 64)
    assert torch.equal(local_gemm.gemm_os_cyclic(A, W), ms.gemm_os(A, pack_slices(W, 5, 8, 0)))


def test_where_the_library_takes_it():
    lib = _lib.load()
    r = lambda *s: torch.randn(*s, device="cuda")
    for call, ids in ((lambda: ms.gemm_os([r(512, 256)] * 4, [r(256, 512)] * 4), {WAVES}), (lambda: ms.gemm_ls(r(256, 1024), [r(256, 1024)] * 4), {WAVES}),
                      (lambda: ms.gemm_os([r(256, 4096)], [r(4096, 256)]), {24}), (lambda: ms.gemm_os([r(2048, 1024)], [r(1024, 2048)]), set(range(21, 28)))):
        call()
        assert lib.ms_query(_lib.MS_QUERY_LAST_VARIANT) in ids
    assert lib.ms_set_variant(WAVES + 200) == _lib.MS_ERR_ARG
    lib.ms_set_variant(0)
