"""Global products of the ring algorithms, which run the devices of a mesh column (OS) or the whole mesh (LS, RS) in one launch: the values of the
same products device by device, and what the bodies refuse."""
import pytest
import torch

from meshslice_amd import TensorParallel as TP
from meshslice_amd.mesh import Mesh, create_device_mesh

pytestmark = pytest.mark.gpu


def _pair(flow, m, n, k, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    R = lambda r, c: torch.randn(r, c, generator=g, device="cuda").to(dtype)
    return (R(k, m) if flow == "rs" else R(m, k)), (R(n, k) if flow == "ls" else R(k, n))


def _device_by_device(f, X, W, monkeypatch):
    with monkeypatch.context() as mp:
        mp.setattr(TP, "_fits_whole_mesh", lambda *a: False)
        return f(X, W)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("algorithm,R,C", [("wang", 1, 2), ("wang", 2, 4), ("wang", 4, 2), ("wang", 1, 3), ("wang", 3, 1), ("cannon", 2, 2), ("cannon", 3, 3)])
def test_ring_products_of_the_whole_mesh(algorithm, R, C, flow, dtype, monkeypatch):
    """LS and RS: the same bits.  OS in bf16 the same bits too where neither way splits its contraction (K is below two K steps a part here, and the fp32
    tiles add in one order); fp32 may share the contraction out over waves on one way only: both then lie within the roundings of k additions."""
    q = 2 * R * C * 8
    for m, n, k, pad in [(q, q, q, 0), (3 * q, q, 2 * q, 0), (q, 2 * q, q, 8)]:
        X, W = _pair(flow, m, n, k, dtype)
        if pad:      # (rows further apart than they are long)
            X, W = (torch.cat([t, t[:, :pad]], 1)[:, :t.shape[1]] for t in (X, W))
            assert X.stride(0) == X.shape[1] + pad
        f = getattr(TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), algorithm), flow.upper())()
        got, want = f(X, W), _device_by_device(f, X, W, monkeypatch)
        if flow != "os" or dtype == torch.bfloat16:
            assert torch.equal(got, want)
        else:
            assert float((got.double() - want.double()).norm() / want.double().norm()) <= 2.0 ** -22 * k ** 0.5


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
def test_rows_that_overlap_and_odd_bases_are_copied(flow, monkeypatch):
    f = getattr(TP.SPMD(Mesh(create_device_mesh((2, 2)), ("row", "col")), "wang"), flow.upper())()
    X, W = _pair(flow, 64, 64, 64, torch.bfloat16)
    flat = torch.randn(64 * 72 + 1, device="cuda").bfloat16()
    for x in (flat[1:].as_strided((64, 64), (72, 1)), flat.as_strided((64, 64), (40, 1))):
        assert torch.equal(f(x, W), _device_by_device(f, x, W, monkeypatch))
        assert torch.equal(f(X, x), _device_by_device(f, X, x, monkeypatch))


def test_what_the_ring_bodies_refuse_stays_refused():
    f = TP.SPMD(Mesh(create_device_mesh((1, 2)), ("row", "col")), "wang")
    X, W = _pair("os", 32, 32, 24, torch.bfloat16)       # half-blocks of six contraction elements
    with pytest.raises(ValueError, match="must be multiples of 8"):
        f.OS()(X, W)
    X, W = _pair("ls", 32, 2 * 2 * 2, 32, torch.bfloat16)      # half-blocks of two output columns
    with pytest.raises(ValueError, match="are not 16-byte aligned|must be multiples of"):
        f.LS()(X, W)


@pytest.mark.parametrize("flow", ["os", "ls", "rs"])
@pytest.mark.parametrize("algorithm", ["wang", "cannon"])
def test_which_products_run_at_once(algorithm, flow, monkeypatch):
    """All but Cannon's OS do without the bodies of single devices, and operands whose half-blocks do not fit are left to those."""
    f = getattr(TP.SPMD(Mesh(create_device_mesh((2, 2)), ("row", "col")), algorithm), flow.upper())()
    X, W = _pair(flow, 64, 64, 64, torch.bfloat16)
    want = f(X, W)

    class ADevice(Exception):
        pass

    def body(*a):
        raise ADevice
    for name in ("_ring_os", "_ring_ls", "_ring_rs"):
        monkeypatch.setattr(TP, name, body)
    if (algorithm, flow) == ("cannon", "os"):
        with pytest.raises(ADevice):
            f(X, W)
    else:
        assert torch.equal(f(X, W), want)
    rows = torch.randn(64 * 72, device="cuda").bfloat16().as_strided((64, 64), (40, 1))
    with pytest.raises(ADevice):
        f(rows, W)
    with pytest.raises(ADevice):
        f(X, rows)


@pytest.mark.parametrize("R,C", [(1, 2), (2, 2), (4, 1), (1, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_column_blocks_are_written_in_place_only_where_they_are_large(R, C, dtype, monkeypatch):
    """A call with out= costs the host 15 us more: 1x2 devices of small layers took 1.4 of the time device by device with it."""
    f = TP.SPMD(Mesh(create_device_mesh((R, C)), ("row", "col")), "wang").OS()
    X, W = _pair("os", 64, 64, 64, dtype)
    outs, real = [], TP.local_gemm.gemm_os
    monkeypatch.setattr(TP.local_gemm, "gemm_os", lambda a, b, out=None: (outs.append(out), real(a, b, out=out))[1])
    copied = f(X, W)
    assert outs == [None] * C
    monkeypatch.setattr(TP, "RING_IN_PLACE_BYTES", 0)
    assert torch.equal(f(X, W), copied) and len(outs) == 2 * C and all((o is None) == (C == 1) for o in outs[C:])
    assert torch.equal(copied, _device_by_device(f, X, W, monkeypatch))
