"""The per-device local contraction of the three dataflows on torch device tensors.

These functions are what the per-device bodies in TensorParallel.py call where the reference calls
``jnp.einsum`` / ``@`` (reference TensorParallel.py:22,26,31,162,167,172,181,187,203,209).  torch is
used only to own device memory and to name the current stream; all arithmetic happens in
libmeshslice_hip.so.
"""
from __future__ import annotations

import contextlib
import ctypes
import threading
from typing import List, Optional, Sequence

import torch

from . import _lib

_DT = {torch.float32: _lib.MS_DTYPE_F32, torch.bfloat16: _lib.MS_DTYPE_BF16}


def _dt(t: torch.Tensor) -> int:
    if t.dtype not in _DT:
        raise TypeError(f"unsupported dtype {t.dtype}: the local GEMM takes float32 or bfloat16")
    return _DT[t.dtype]


def _check2d(t: torch.Tensor, name: str) -> None:
    if not t.is_cuda:
        raise _lib.MeshSliceError(f"{name} is not on the GPU: the local GEMM has no CPU path")
    if t.dim() != 2 or t.stride(1) != 1:
        raise ValueError(f"{name} must be a row-major 2-D tensor (got shape {tuple(t.shape)}, strides {t.stride()})")


def _stream() -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _same(ts: Sequence[torch.Tensor], name: str):
    if len(ts) < 1:
        raise ValueError(f"{name}: need at least one slice")
    s0 = ts[0]
    _check2d(s0, name)
    shape, strides, dtype, device = s0.shape, s0.stride(), s0.dtype, s0.device
    for t in ts:
        if t.shape != shape or t.stride() != strides or t.dtype != dtype or t.device != device:
            _check2d(t, name)
            raise ValueError(f"{name}: all slices must share shape, dtype, leading dimension and device")
    return s0


# The ordinary case of a call (plain GPU tensors, output left to the call) is taken by the native call path as a whole
# (_lib.host, csrc/ms_host.cpp); it returns None for everything else, which the functions below then handle or refuse.
# gemm_os of four slices of 512 x 256 x 512 in fp32 takes the host 18.8 us a call without it and 5.5 with it, launch included; one device of a
# 2x4 mesh (gather and LS product) 76 and 27; a training step of 512 x 256 x 1024 on a 4x2 mesh, whose sums are one launch each, 232 and 135.
_HERE = contextlib.nullcontext()


def _on(device: torch.device):
    """``torch.cuda.device(device)``, without its two device switches where the device is the current one already."""
    return _HERE if torch.cuda.current_device() == device.index else torch.cuda.device(device)


_workspaces = {}            # (device index, stream handle) -> uint8 tensor; the native call path holds them too and knows when each was used last
_workspaces_lock = threading.Lock()
_WORKSPACE_CACHE_MAX = 8      # streams per device that keep a workspace of their own (about 100 MB each)


def workspace(device, stream=None) -> torch.Tensor:
    """The split-contraction workspace of ``(device, stream)`` (a uint8 tensor of ``ms_workspace_bytes()`` bytes,
    allocated and prepared with ``ms_workspace_init`` on first use, then kept): ``gemm_os`` hands it to
    ``ms_gemm_os_ws`` so that products with few output tiles can spread their contraction over the idle compute units.

    Calls that share a workspace must not overlap on the device (they share its arrival counters and partial tiles).
    Work on ONE stream never overlaps, so every stream gets a workspace of its own (``stream`` defaults to the current
    one): calls issued from several host threads or on several streams cannot meet in one.  At most
    ``_WORKSPACE_CACHE_MAX`` streams per device keep one; a further stream evicts the least recently used, after
    waiting for the device to finish what is queued (the evicted stream may still be running a product on it).

    While a ``torch.cuda.graph`` capture is under way on the current stream the workspace is allocated inside the capture
    (from the graph's own memory pool, so it lives as long as the graph and later captured calls of the same graph
    reuse it), prepared by a captured fill kernel and not kept here: a graph's replays never share counters with eager
    calls or with another graph's."""
    device = torch.device(device)
    idx = device.index if device.index is not None else torch.cuda.current_device()
    if stream is None:
        stream = torch.cuda.current_stream(idx)
    key = (idx, int(stream.cuda_stream))
    capturing = torch.cuda.is_current_stream_capturing()
    if not capturing:
        with _workspaces_lock:
            ws = _workspaces.get(key)
            if ws is not None:
                _lib.host.workspace_touch(*key)
                return ws
    lib = _lib.load()
    with torch.cuda.device(idx), torch.cuda.stream(stream):
        nbytes = int(lib.ms_workspace_bytes())
        if nbytes <= 0:
            raise _lib.MeshSliceError("could not size the workspace: " + _lib.last_error())
        ws = torch.empty(nbytes, dtype=torch.uint8, device=torch.device("cuda", idx))
        _lib.check(lib.ms_workspace_init(ctypes.c_void_p(ws.data_ptr()), nbytes, ctypes.c_void_p(stream.cuda_stream)))
    if capturing:
        return ws
    with _workspaces_lock:
        have = _workspaces.setdefault(key, ws)      # (another thread on the same stream may have been faster)
        mine = sorted((k for k in _workspaces if k[0] == idx and k != key), key=lambda k: _lib.host.workspace_touch(*k, False))
        drop = mine[:max(0, len(mine) + 1 - _WORKSPACE_CACHE_MAX)]
        for k in drop:      # (the native call path must not hand one out that is about to go)
            _lib.host.workspace_drop(*k)
        evicted = [_workspaces.pop(k) for k in drop]
        _lib.host.workspace_set(*key, have)
    if evicted:
        torch.cuda.synchronize(idx)     # their streams may still be running products that use them
        del evicted
    return have


def _ws_args(device):
    """(pointer, bytes, tensor): the caller keeps the tensor until its call has been issued"""
    ws = workspace(device)
    return ctypes.c_void_p(ws.data_ptr()), ws.numel(), ws


class _Call:
    """One validated local contraction: the C entry points' argument list up to (not including) ``stream``,
    the device it runs on, the output it writes and the Python objects that keep the pointer tables alive."""

    def __init__(self, device, args, out, keep):
        self.device, self.args, self.out, self.keep = device, args, out, keep


def _prepare_os(A_slices, B_slices, out, out_dtype) -> _Call:
    a0 = _same(A_slices, "A_slices"); b0 = _same(B_slices, "B_slices")
    if len(A_slices) != len(B_slices):
        raise ValueError("A_slices and B_slices differ in length")
    if a0.shape[1] != b0.shape[0] or a0.dtype != b0.dtype or a0.device != b0.device:
        raise ValueError(f"slice shapes do not contract: {tuple(a0.shape)} @ {tuple(b0.shape)}")
    m, k = a0.shape; n = b0.shape[1]
    if out is None:
        out = torch.empty((m, n), dtype=out_dtype or a0.dtype, device=a0.device)
    _check2d(out, "out")
    if tuple(out.shape) != (m, n) or out.device != a0.device:
        raise ValueError("out has the wrong shape or device")
    pa, _ka = _lib.ptr_array([t.data_ptr() for t in A_slices])
    pb, _kb = _lib.ptr_array([t.data_ptr() for t in B_slices])
    args = (pa, pb, len(A_slices), m, n, k, a0.stride(0), b0.stride(0),
            ctypes.c_void_p(out.data_ptr()), out.stride(0), _dt(a0), _dt(out))
    return _Call(a0.device, args, out, (_ka, _kb))


def _chunk_views(buf: torch.Tensor):
    """The [rows, columns] parts of a fresh 3-D buffer and their addresses."""
    step, base = buf.stride(0) * buf.element_size(), buf.data_ptr()
    return [buf.select(0, s) for s in range(buf.shape[0])], [base + s * step for s in range(buf.shape[0])]


def _prepare_ls(A, W_slices, out, out_dtype) -> _Call:
    _check2d(A, "A"); w0 = _same(W_slices, "W_slices")
    if A.shape[1] != w0.shape[1] or A.dtype != w0.dtype or A.device != w0.device:
        raise ValueError(f"shapes do not contract: {tuple(A.shape)} @ {tuple(w0.shape)}^T")
    m, k = A.shape; ns = w0.shape[0]; S = len(W_slices)
    dt = _chunk_dtype(out, out_dtype)
    if out is None:
        out, ptrs = _chunk_views(torch.empty((S, m, ns), dtype=dt, device=A.device))
        o0 = out[0]
    else:
        o0 = _same(out, "out")
        if len(out) != S or tuple(o0.shape) != (m, ns) or o0.dtype not in (torch.float32, torch.bfloat16) or o0.device != A.device:
            raise ValueError("out must be S fp32 or bf16 chunks of shape [m, n_slice] on the operands' device")
        ptrs = [t.data_ptr() for t in out]
    pw, _kw = _lib.ptr_array([t.data_ptr() for t in W_slices])
    py, _ky = _lib.ptr_array(ptrs)
    args = (ctypes.c_void_p(A.data_ptr()), A.stride(0), pw, w0.stride(0), S, m, ns, k, py, o0.stride(0), _dt(A), _dt(o0))
    return _Call(A.device, args, list(out), (_kw, _ky))


def _prepare_rs(X_slices, W, out, out_dtype) -> _Call:
    _check2d(W, "W"); x0 = _same(X_slices, "X_slices")
    if x0.shape[0] != W.shape[0] or x0.dtype != W.dtype or x0.device != W.device:
        raise ValueError(f"shapes do not contract: {tuple(x0.shape)}^T @ {tuple(W.shape)}")
    k, ms = x0.shape; n = W.shape[1]; S = len(X_slices)
    dt = _chunk_dtype(out, out_dtype)
    if out is None:
        out, ptrs = _chunk_views(torch.empty((S, ms, n), dtype=dt, device=W.device))
        o0 = out[0]
    else:
        o0 = _same(out, "out")
        if len(out) != S or tuple(o0.shape) != (ms, n) or o0.dtype not in (torch.float32, torch.bfloat16) or o0.device != W.device:
            raise ValueError("out must be S fp32 or bf16 chunks of shape [m_slice, n] on the operands' device")
        ptrs = [t.data_ptr() for t in out]
    px, _kx = _lib.ptr_array([t.data_ptr() for t in X_slices])
    py, _ky = _lib.ptr_array(ptrs)
    args = (px, x0.stride(0), ctypes.c_void_p(W.data_ptr()), W.stride(0), S, ms, n, k, py, o0.stride(0), _dt(W), _dt(o0))
    return _Call(W.device, args, list(out), (_kx, _ky))


def gemm_os(A_slices: Sequence[torch.Tensor], B_slices: Sequence[torch.Tensor],
            out: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None,
            activation: Optional[str] = None, residual: Optional[torch.Tensor] = None,
            row_moments=None) -> torch.Tensor:
    """``C = sum_s A_s @ B_s`` with fp32 accumulation over all slices, rounded once.

    Optional fused epilogue (bf16 operands): ``C = act(sum) + residual`` with ``activation='gelu'`` (tanh
    form) and ``residual`` of C's shape and dtype; ``row_moments=(row_sum, row_sumsq)`` are fp32 vectors of
    length m (either may be None) to which the row sums / sums of squares of the fp32 result are ADDED."""
    if out is None and row_moments is None and activation in (None, "gelu"):
        y = _lib.host.gemm_os(A_slices, B_slices, out_dtype, activation is not None, residual)
        if y is not None:
            return y
    call = _prepare_os(A_slices, B_slices, out, out_dtype)
    out = call.out
    m, n = out.shape
    if activation not in (None, "gelu"):
        raise ValueError(f"unknown activation {activation!r} (None or 'gelu')")
    res_ptr, ldr = None, 0
    if residual is not None:
        _check2d(residual, "residual")
        if tuple(residual.shape) != (m, n) or residual.dtype != out.dtype or residual.device != out.device:
            raise ValueError("residual must have the shape, dtype and device of the output")
        res_ptr, ldr = ctypes.c_void_p(residual.data_ptr()), residual.stride(0)
    moments = [None, None]
    for idx, t in enumerate(row_moments or (None, None)):
        if t is not None:
            if not (t.is_cuda and t.dtype == torch.float32 and t.dim() == 1 and t.numel() == m and t.is_contiguous()
                    and t.device == out.device):
                raise ValueError("row moments must be contiguous fp32 GPU vectors of length m on the output's device")
            moments[idx] = ctypes.c_void_p(t.data_ptr())
    with _on(call.device):
        stream = torch.cuda.current_stream()
        ws = workspace(call.device, stream)
        rc = _lib.load().ms_gemm_os_ws(*call.args,
                                       _lib.MS_ACT_GELU if activation == "gelu" else _lib.MS_ACT_NONE,
                                       res_ptr, ldr, moments[0], moments[1], ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                                       ctypes.c_void_p(stream.cuda_stream))
    _lib.check(rc)
    return out


def gemm_os_cyclic(A_slices: Sequence[torch.Tensor], W: torch.Tensor) -> torch.Tensor:
    """``gemm_os`` on the block-cyclic row slices of W (blocks of eight rows), read where they lie (``ms_gemm_os_cyclic``): the
    bits of ``gemm_os(A_slices, pack_slices(W, len(A_slices), 8, 0))`` without that copy."""
    y = _lib.host.gemm_os_cyclic(A_slices, W)
    if y is not None:
        return y
    a0 = _same(A_slices, "A_slices"); _check2d(W, "W")
    S = len(A_slices)
    if S * a0.shape[1] != W.shape[0] or a0.dtype != W.dtype or a0.device != W.device:
        raise ValueError(f"shapes do not contract: {S} slices {tuple(a0.shape)} @ {tuple(W.shape)}")
    m, k = a0.shape; n = W.shape[1]
    out = torch.empty((m, n), dtype=W.dtype, device=W.device)
    pa, _ka = _lib.ptr_array([t.data_ptr() for t in A_slices])
    with _on(W.device):
        stream = torch.cuda.current_stream()
        ws = workspace(W.device, stream)
        rc = _lib.load().ms_gemm_os_cyclic(pa, ctypes.c_void_p(W.data_ptr()), S, m, n, k, a0.stride(0), W.stride(0), ctypes.c_void_p(out.data_ptr()), n,
                                           _dt(W), _dt(W), ctypes.c_void_p(ws.data_ptr()), ws.numel(), ctypes.c_void_p(stream.cuda_stream))
    _lib.check(rc)
    return out


def _chunk_dtype(out, out_dtype):
    """dtype of the LS / RS chunks: that of ``out`` if given, else ``out_dtype``, else fp32."""
    if out is not None and len(out) > 0:
        if out_dtype is not None and out[0].dtype != out_dtype:
            raise ValueError("out_dtype contradicts the dtype of out")
        return out[0].dtype
    dt = torch.float32 if out_dtype is None else out_dtype
    if dt not in (torch.float32, torch.bfloat16):
        raise ValueError("chunks are fp32 or bf16")
    return dt


def gemm_os_gated(A_slices: Sequence[torch.Tensor], B_slices: Sequence[torch.Tensor], slice_ready: torch.Tensor,
                  out: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None,
                  timeout_ms: int = 2000) -> torch.Tensor:
    """gemm_os as ONE launch that may be enqueued before its slices have arrived (``ms_gemm_os_gated``): the kernel
    reads slice s of A and of B only after ``slice_ready[s]`` has become non-zero, the way the reference's
    output-stationary body multiplies slice k while slice k + 1 is still being gathered (MeshFlow_OS,
    TensorParallel.py:163-171).  ``slice_ready`` is an int32 GPU tensor of S + 1 words: the flags (set them with
    ``signal_set`` on the stream that fills the slice, after the fill) and, last, a status word that must be zero before
    the call and reads 1 afterwards if a wait lasted longer than ``timeout_ms`` (the result is then void: check it with
    ``gate_timed_out`` once the stream has been synchronised).  A producer that needs compute units of this device
    only runs beside the waiting product when units have been reserved (``ms_set_reserved_cus``)."""
    call = _prepare_os(A_slices, B_slices, out, out_dtype)
    _check_flags(slice_ready, len(A_slices), call.device)
    ws_ptr, ws_bytes, _ws_keep = _ws_args(call.device)
    with _on(call.device):
        rc = _lib.load().ms_gemm_os_gated(*call.args, ws_ptr, ws_bytes, ctypes.c_void_p(slice_ready.data_ptr()),
                                          int(timeout_ms), _stream())
    _lib.check(rc)
    return call.out


def _check_flags(slice_ready, S, device):
    if not (isinstance(slice_ready, torch.Tensor) and slice_ready.is_cuda and slice_ready.dtype == torch.int32
            and slice_ready.dim() == 1 and slice_ready.numel() == S + 1 and slice_ready.is_contiguous()
            and slice_ready.device == device):
        raise ValueError("slice_ready must be a contiguous int32 GPU tensor of S + 1 words on the operands' device")


def _chunks_gated(entry, call, S, slice_ready, chunk_done, timeout_ms):
    _check_flags(slice_ready, S, call.device)
    tiles = ctypes.c_int(0)
    if chunk_done is not None:
        _check_counters(chunk_done, S, call.device)
    with _on(call.device):
        rc = entry(*call.args, ctypes.c_void_p(chunk_done.data_ptr()) if chunk_done is not None else None,
                   ctypes.byref(tiles) if chunk_done is not None else None,
                   ctypes.c_void_p(slice_ready.data_ptr()), int(timeout_ms), _stream())
    _lib.check(rc)
    return call.out if chunk_done is None else (call.out, tiles.value)


def gemm_ls_gated(A: torch.Tensor, W_slices: Sequence[torch.Tensor], slice_ready: torch.Tensor,
                  out: Optional[List[torch.Tensor]] = None, out_dtype: Optional[torch.dtype] = None,
                  chunk_done: Optional[torch.Tensor] = None, timeout_ms: int = 2000):
    """gemm_ls as one launch that may be enqueued before the weight slices have arrived (``ms_gemm_ls_gated``): ``W_s`` is
    read only after ``slice_ready[s]`` has become non-zero (MeshFlow_LS gathers slice k + 1 while chunk k is multiplied,
    TensorParallel.py:176-189); flags, status word and time limit as for ``gemm_os_gated``.  With ``chunk_done`` (see
    ``gemm_ls_signal``) the call also counts finished tiles per chunk and returns ``(chunks, tiles_per_chunk)``."""
    return _chunks_gated(_lib.load().ms_gemm_ls_gated, _prepare_ls(A, W_slices, out, out_dtype), len(W_slices), slice_ready, chunk_done, timeout_ms)


def gemm_rs_gated(X_slices: Sequence[torch.Tensor], W: torch.Tensor, slice_ready: torch.Tensor,
                  out: Optional[List[torch.Tensor]] = None, out_dtype: Optional[torch.dtype] = None,
                  chunk_done: Optional[torch.Tensor] = None, timeout_ms: int = 2000):
    """gemm_rs behind the input gate (``ms_gemm_rs_gated``; see gemm_ls_gated; reference TensorParallel.py:198-212):
    ``X_s`` is read only after ``slice_ready[s]`` has become non-zero."""
    return _chunks_gated(_lib.load().ms_gemm_rs_gated, _prepare_rs(X_slices, W, out, out_dtype), len(X_slices), slice_ready, chunk_done, timeout_ms)


def signal_set(flags: torch.Tensor, index: int, value: int = 1) -> None:
    """``flags[index] = value`` on the current stream, after everything enqueued on it before, as a release at system
    scope (``ms_signal_set``): the producer's half of the gated calls."""
    if not (isinstance(flags, torch.Tensor) and flags.is_cuda and flags.dtype == torch.int32 and flags.dim() == 1 and flags.is_contiguous()):
        raise ValueError("flags must be a contiguous int32 GPU vector")
    if not 0 <= index < flags.numel():
        raise IndexError(f"flag index {index} outside [0, {flags.numel()})")
    with torch.cuda.device(flags.device):
        rc = _lib.load().ms_signal_set(ctypes.c_void_p(flags.data_ptr() + 4 * index), int(value), _stream())
    _lib.check(rc)


def gate_timed_out(slice_ready: torch.Tensor) -> bool:
    """Whether a gated call with these flags gave up waiting for a slice (synchronises with the device)."""
    return bool(slice_ready[-1].item() != 0)


def gemm_ls(A: torch.Tensor, W_slices: Sequence[torch.Tensor],
            out: Optional[List[torch.Tensor]] = None, out_dtype: Optional[torch.dtype] = None) -> List[torch.Tensor]:
    """``Y_s = A @ W_s^T``, W_s stored ``[n_slice, k]``.  Chunks are fp32 by default (exact partial sums for
    the reduce-scatter); ``out_dtype=torch.bfloat16`` gives what the reference's einsum returns for bf16
    operands (TensorParallel.py:181-189): one rounding of the fp32 accumulator, half the bytes."""
    if out is None:
        chunks = _lib.host.gemm_ls(A, W_slices, out_dtype)
        if chunks is not None:
            return chunks
    call = _prepare_ls(A, W_slices, out, out_dtype)
    with _on(call.device):
        rc = _lib.load().ms_gemm_ls_ex(*call.args, _stream())
    _lib.check(rc)
    return call.out


def gemm_rs(X_slices: Sequence[torch.Tensor], W: torch.Tensor,
            out: Optional[List[torch.Tensor]] = None, out_dtype: Optional[torch.dtype] = None) -> List[torch.Tensor]:
    """``Y_s = X_s^T @ W``, X_s stored ``[k, m_slice]``; chunks fp32 by default, bf16 on request (see gemm_ls)."""
    if out is None:
        chunks = _lib.host.gemm_rs(X_slices, W, out_dtype)
        if chunks is not None:
            return chunks
    call = _prepare_rs(X_slices, W, out, out_dtype)
    with _on(call.device):
        rc = _lib.load().ms_gemm_rs_ex(*call.args, _stream())
    _lib.check(rc)
    return call.out


def gemm_ls_cyclic(A: torch.Tensor, W: torch.Tensor, S: int) -> List[torch.Tensor]:
    """``gemm_ls`` on the S block-cyclic row slices of W (blocks of eight rows), read where they lie (``ms_gemm_ls_cyclic``): the fp32
    chunks of ``gemm_ls(A, pack_slices(W, S, 8, 0))`` without that copy."""
    chunks = _lib.host.gemm_ls_cyclic(A, W, S)
    if chunks is not None:
        return chunks
    _check2d(A, "A"); _check2d(W, "W")
    if S < 1 or W.shape[0] % S or A.shape[1] != W.shape[1] or A.dtype != W.dtype or A.device != W.device:
        raise ValueError(f"shapes do not contract: {tuple(A.shape)} @ {S} row slices of {tuple(W.shape)}^T")
    m, k = A.shape; n = W.shape[0] // S
    out, ptrs = _chunk_views(torch.empty((S, m, n), dtype=torch.float32, device=A.device))
    py, _ky = _lib.ptr_array(ptrs)
    with _on(A.device):
        rc = _lib.load().ms_gemm_ls_cyclic(ctypes.c_void_p(A.data_ptr()), A.stride(0), ctypes.c_void_p(W.data_ptr()), W.stride(0), S, m, n, k, py, n,
                                           _dt(A), _dt(out[0]), _stream())
    _lib.check(rc)
    return out


def gemm_ls_peers(A_shards: Sequence[torch.Tensor], W_slices_by_peer: Sequence[Sequence[torch.Tensor]]) -> List[List[torch.Tensor]]:
    """``gemm_ls`` of the P devices of a mesh row in one launch (``ms_gemm_ls_peers``): fp32 chunks
    ``[p][s] = A_shards[p] @ W_slices_by_peer[p][s]^T``, all shards and all slices of one shape and leading dimension."""
    a0 = _same(A_shards, "A_shards")
    flat = [w for peer in W_slices_by_peer for w in peer]
    w0 = _same(flat, "W_slices")
    P, S = len(A_shards), len(flat) // len(A_shards)
    if any(len(peer) != S for peer in W_slices_by_peer) or len(W_slices_by_peer) != P:
        raise ValueError("every device must bring the same number of slices")
    if a0.shape[1] != w0.shape[1] or a0.dtype != w0.dtype or a0.device != w0.device:
        raise ValueError(f"shapes do not contract: {tuple(a0.shape)} @ {tuple(w0.shape)}^T")
    m, k = a0.shape; ns = w0.shape[0]
    return _peers(_lib.load().ms_gemm_ls_peers, A_shards, flat, P, S, (m, ns), (m, ns, k))


def gemm_rs_peers(X_slices_by_peer: Sequence[Sequence[torch.Tensor]], W_shards: Sequence[torch.Tensor]) -> List[List[torch.Tensor]]:
    """``gemm_rs`` of the P devices of a mesh column in one launch (``ms_gemm_rs_peers``): fp32 chunks
    ``[p][s] = X_slices_by_peer[p][s]^T @ W_shards[p]``."""
    w0 = _same(W_shards, "W_shards")
    flat = [x for peer in X_slices_by_peer for x in peer]
    x0 = _same(flat, "X_slices")
    P, S = len(W_shards), len(flat) // len(W_shards)
    if any(len(peer) != S for peer in X_slices_by_peer) or len(X_slices_by_peer) != P:
        raise ValueError("every device must bring the same number of slices")
    if x0.shape[0] != w0.shape[0] or x0.dtype != w0.dtype or x0.device != w0.device:
        raise ValueError(f"shapes do not contract: {tuple(x0.shape)}^T @ {tuple(w0.shape)}")
    k, ms = x0.shape; n = w0.shape[1]
    return _peers(_lib.load().ms_gemm_rs_peers, flat, W_shards, P, S, (ms, n), (ms, n, k))


def _peers(entry, first, second, P, S, chunk, extents):
    f0, s0 = first[0], second[0]
    buf = torch.empty((P * S,) + chunk, dtype=torch.float32, device=f0.device)
    pf, _kf = _lib.ptr_array([t.data_ptr() for t in first])
    ps, _ks = _lib.ptr_array([t.data_ptr() for t in second])
    chunks, ptrs = _chunk_views(buf)
    py, _ky = _lib.ptr_array(ptrs)
    with _on(f0.device):
        rc = entry(pf, f0.stride(0), ps, s0.stride(0), P, S, *extents, py, chunk[1], _dt(f0), _lib.MS_DTYPE_F32, _stream())
    _lib.check(rc)
    return [chunks[p * S:(p + 1) * S] for p in range(P)]


def gemm_ls_sum(X: torch.Tensor, W: torch.Tensor, P: int) -> torch.Tensor:
    """``X @ W^T`` as the P devices of a mesh row compute it between them (``ms_gemm_ls_sum``): the contraction in P equal
    windows, each window's partial sum in fp32 by itself, the partial sums added up in window order and rounded once.  bf16."""
    y = _lib.host.gemm_ls_sum(X, W, P)
    if y is not None:
        return y
    _check2d(X, "X"); _check2d(W, "W")
    if X.shape[1] != W.shape[1] or X.dtype != W.dtype or X.device != W.device or X.shape[1] % P:
        raise ValueError(f"shapes do not contract in {P} windows: {tuple(X.shape)} @ {tuple(W.shape)}^T")
    step = X.shape[1] // P * X.element_size()
    return _sum(_lib.load().ms_gemm_ls_sum, X, W, P, step, step, X.shape[0], W.shape[0], X.shape[1] // P)


def gemm_rs_sum(X: torch.Tensor, W: torch.Tensor, P: int) -> torch.Tensor:
    """``X^T @ W`` in the same way (``ms_gemm_rs_sum``): the P windows are those of the devices of a mesh column."""
    y = _lib.host.gemm_rs_sum(X, W, P)
    if y is not None:
        return y
    _check2d(X, "X"); _check2d(W, "W")
    if X.shape[0] != W.shape[0] or X.dtype != W.dtype or X.device != W.device or X.shape[0] % P:
        raise ValueError(f"shapes do not contract in {P} windows: {tuple(X.shape)}^T @ {tuple(W.shape)}")
    k = X.shape[0] // P
    return _sum(_lib.load().ms_gemm_rs_sum, X, W, P, k * X.stride(0) * X.element_size(), k * W.stride(0) * W.element_size(), X.shape[1], W.shape[1], k)


def prefers_sum(flow: str, P: int, S: int, m: int, n: int, k: int) -> bool:
    """Whether the sum over a mesh line of P devices, k contraction elements each, is expected sooner from gemm_ls_sum / gemm_rs_sum than from
    fp32 chunks of S slices added up in memory (``ms_prefers_sum``)."""
    pays = _lib.host.prefers_sum(flow == "rs", P, S, m, n, k)
    return bool(_lib.load().ms_prefers_sum(flow == "rs", P, S, m, n, k)) if pays is None else pays


def _sum(entry, X, W, P, x_step, w_step, m, n, k):
    out = torch.empty((m, n), dtype=X.dtype, device=X.device)
    x0, w0 = X.data_ptr(), W.data_ptr()
    px, _kx = _lib.ptr_array([x0 + p * x_step for p in range(P)])
    pw, _kw = _lib.ptr_array([w0 + p * w_step for p in range(P)])
    with _on(X.device):
        stream = torch.cuda.current_stream()
        ws = workspace(X.device, stream)
        rc = entry(px, X.stride(0), pw, W.stride(0), P, m, n, k, ctypes.c_void_p(out.data_ptr()), n, _dt(X), _dt(out),
                   ctypes.c_void_p(ws.data_ptr()), ws.numel(), ctypes.c_void_p(stream.cuda_stream))
    _lib.check(rc)
    return out


def _check_counters(chunk_done: torch.Tensor, S: int, device) -> None:
    if not (isinstance(chunk_done, torch.Tensor) and chunk_done.is_cuda and chunk_done.device == device
            and chunk_done.dtype == torch.int32 and chunk_done.is_contiguous() and chunk_done.numel() >= S):
        raise ValueError(f"chunk_done must be a contiguous int32 tensor of at least {S} counters on {device}")


def gemm_ls_signal(A: torch.Tensor, W_slices: Sequence[torch.Tensor], chunk_done: torch.Tensor,
                   out: Optional[List[torch.Tensor]] = None, out_dtype: Optional[torch.dtype] = None):
    """gemm_ls with per-chunk completion counters (``ms_gemm_ls_signal``): the kernel adds 1 to ``chunk_done[s]``
    (int32, zero before the call) after each output tile of ``Y_s`` is in memory, so that the reduce-scatter of chunk
    s (reference TensorParallel.py:182-189) can start before the call has ended.  Returns ``(chunks, tiles_per_chunk)``:
    ``Y_s`` is complete when ``chunk_done[s] == tiles_per_chunk``."""
    call = _prepare_ls(A, W_slices, out, out_dtype)
    _check_counters(chunk_done, len(W_slices), call.device)
    tiles = ctypes.c_int(0)
    with _on(call.device):
        rc = _lib.load().ms_gemm_ls_signal(*call.args, ctypes.c_void_p(chunk_done.data_ptr()), ctypes.byref(tiles), _stream())
    _lib.check(rc)
    return call.out, tiles.value


def gemm_rs_signal(X_slices: Sequence[torch.Tensor], W: torch.Tensor, chunk_done: torch.Tensor,
                   out: Optional[List[torch.Tensor]] = None, out_dtype: Optional[torch.dtype] = None):
    """gemm_rs with per-chunk completion counters (``ms_gemm_rs_signal``, see gemm_ls_signal; reference
    TensorParallel.py:204-212)."""
    call = _prepare_rs(X_slices, W, out, out_dtype)
    _check_counters(chunk_done, len(X_slices), call.device)
    tiles = ctypes.c_int(0)
    with _on(call.device):
        rc = _lib.load().ms_gemm_rs_signal(*call.args, ctypes.c_void_p(chunk_done.data_ptr()), ctypes.byref(tiles), _stream())
    _lib.check(rc)
    return call.out, tiles.value


def time_call(flow: str, operands, out, warmup: int = 5, reps: int = 20) -> List[float]:
    """Per-launch milliseconds (HIP events on the current stream) of one local contraction.

    ``flow`` is 'os', 'ls' or 'rs'; ``operands`` / ``out`` are what gemm_os / gemm_ls / gemm_rs take (``out`` is
    required here) and are checked the same way; LS / RS chunks may be fp32 or bf16."""
    if flow not in ("os", "ls", "rs"):
        raise ValueError(f"unknown dataflow {flow!r}")
    if out is None:
        raise ValueError("time_call needs the output buffer(s)")
    if int(warmup) < 0 or int(reps) < 1:
        raise ValueError("time_call needs warmup >= 0 and reps >= 1")
    first, second = operands
    lib = _lib.load()
    if flow == "os":
        call = _prepare_os(first, second, out, None)
        ms = (ctypes.c_float * int(reps))()
        ws_ptr, ws_bytes, _ws_keep = _ws_args(call.device)
        with _on(call.device):
            rc = lib.ms_time_os_ws(*call.args, ws_ptr, ws_bytes, _stream(), int(warmup), int(reps), ms)
        _lib.check(rc)
        return list(ms)
    elif flow == "ls":
        call, fn = _prepare_ls(first, second, out, None), lib.ms_time_ls_ex
    else:
        call, fn = _prepare_rs(first, second, out, None), lib.ms_time_rs_ex
    ms = (ctypes.c_float * int(reps))()
    with _on(call.device):
        rc = fn(*call.args, _stream(), int(warmup), int(reps), ms)
    _lib.check(rc)
    return list(ms)


def mfma_stream_rate(operands: Optional[torch.Tensor] = None, iters: int = 4000, warmup: int = 20, reps: int = 200,
                     shape: str = "32x32x16", waves_per_simd: int = 1) -> float:
    """FLOP/s that the current GPU sustains on a bare stream of one bf16 MFMA instruction
    (``ms_probe_mfma_stream_ex``): the practical ceiling, under the device's power limit, for the operand data
    given (default: N(0,1) values rounded to bf16, seed 0).  ``shape`` is '32x32x16' (the instruction of the
    big-tile kernels) or '16x16x32'; ``waves_per_simd`` 1 or 2.  ``warmup + reps`` launches of about a
    millisecond each, so the figure is the sustained one."""
    shapes = {"32x32x16": _lib.MS_MFMA_32X32X16, "16x16x32": _lib.MS_MFMA_16X16X32}
    if shape not in shapes:
        raise ValueError(f"unknown MFMA shape {shape!r} (one of {sorted(shapes)})")
    if waves_per_simd not in (1, 2):
        raise ValueError("waves_per_simd must be 1 or 2")
    dev = torch.device("cuda", torch.cuda.current_device())
    need = 16 * 64 * 8
    if operands is None:
        g = torch.Generator(device="cpu").manual_seed(0)
        operands = torch.randn(need, generator=g).to(torch.bfloat16).to(dev)
    if not (operands.is_cuda and operands.dtype == torch.bfloat16 and operands.is_contiguous() and operands.numel() >= need):
        raise ValueError(f"operands must be a contiguous bf16 GPU tensor of at least {need} elements")
    with torch.cuda.device(operands.device):
        cus = _lib.load().ms_query(_lib.MS_QUERY_CU_COUNT)
    if cus <= 0:
        raise _lib.MeshSliceError("could not read the compute-unit count of the device")
    sink = torch.empty(256 * waves_per_simd * int(cus), dtype=torch.float32, device=operands.device)
    ms, fl = ctypes.c_float(0.0), ctypes.c_double(0.0)
    with torch.cuda.device(operands.device):
        rc = _lib.load().ms_probe_mfma_stream_ex(ctypes.c_void_p(operands.data_ptr()), ctypes.c_void_p(sink.data_ptr()),
                                                 shapes[shape], int(waves_per_simd), int(iters), int(warmup), int(reps),
                                                 ctypes.byref(ms), ctypes.byref(fl), _stream())
    _lib.check(rc)
    return fl.value / (ms.value * 1e-3)
