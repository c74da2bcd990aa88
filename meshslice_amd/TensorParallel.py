"""2-D tensor-parallel GEMM: the reference's ``SPMD(mesh, algorithm, blocksize).OS/LS/RS(K)`` surface
with the mesh emulated on the host and the local contraction running in hand-written gfx950 kernels.

Mirrors reference TensorParallel.py: the unsliced bodies ``Collective_OS/LS/RS`` (:19-32), the sliced
bodies ``MeshFlow_OS/LS/RS`` (:153-214) and the builder ``SPMD`` (:346-377).  Differences, all forced
by having one GPU and no tracing compiler:

* the callable returned by ``OS/LS/RS`` takes the GLOBAL operands (torch tensors on the GPU), logically
  sharded ``P(row, col)``, and returns the GLOBAL result; the devices' gathers, products and reduce-scatters run in
  one launch each where the shapes allow it (_fits_whole_mesh), else it runs every mesh device's body in turn;
* ``.device(i, j)`` runs ONE device's body and returns what that device produces before any
  cross-device reduction: its output block (OS) or its S fp32 partial chunks (LS / RS);
* all_gather / psum_scatter move data between the emulated devices' buffers on the one GPU: the
  block-cyclic slicing, the placement of gathered slices and the reduce + interleave of the chunks run
  in the layout kernels of libmeshslice_hip.so (slice_layout.py), not in torch indexing;
* the local contraction accumulates in fp32 over all slices and rounds once (the reference carries
  the running sum in the input dtype, :167);
* the sliced OS body rejects ``K == 1``: the reference adds slice 0 twice in that case (:163,:172);
  use ``algorithm='collective'`` for the unsliced product;
* the ring baselines 'wang' and 'cannon' (:34-149, :218-342): one device's body drives the same kernels with 2 * size
  half-block slices in ring order, the hops themselves being host index arithmetic.  A global product takes that order only where it
  shows in the result (OS); the LS and RS bodies hand out Collective's partial sums, and their global products are computed as its are
  (_RING_BODIES), so timing those does not tell the algorithms apart.
"""
from __future__ import annotations

import threading
from typing import Callable, List, Sequence

import torch

from . import local_gemm, slice_layout
from .mesh import Mesh, PartitionSpec as P  # noqa: F401  (re-exported like the reference's imports)


def allclose(a, b) -> bool:
    """The reference's acceptance test (TensorParallel.py:16-17)."""
    return bool(torch.allclose(torch.as_tensor(a).float().cpu(), torch.as_tensor(b).float().cpu(), atol=1e-2, rtol=1e-2))


# ------------------------------------------------------------------------------------------------
# host-side mesh plumbing
# ------------------------------------------------------------------------------------------------

def _shards(G: torch.Tensor, R: int, C: int) -> List[List[torch.Tensor]]:
    """blocks[i][j] = device (i,j)'s shard of a matrix sharded P(row, col) (views, no copies)."""
    if G.dim() != 2:
        raise ValueError("operands must be 2-D")
    if G.shape[0] % R or G.shape[1] % C:
        raise ValueError(f"matrix {tuple(G.shape)} does not shard evenly over a {R}x{C} mesh")
    h, w = G.shape[0] // R, G.shape[1] // C
    return [[G[i * h:(i + 1) * h, j * w:(j + 1) * w] for j in range(C)] for i in range(R)]


class _Line:
    """The shards of one mesh row or column of a global matrix, in axis order: the views, made where they are asked for, and
    the one view that covers them."""

    def __init__(self, panel: torch.Tensor, n: int, axis: int, step=None):
        self.panel, self.n, self.axis, self.step = panel, n, axis, panel.shape[axis] // n if step is None else step

    def __len__(self):
        return self.n

    def __getitem__(self, p):
        if not -self.n <= p < self.n:
            raise IndexError(p)
        return self.panel.narrow(self.axis, p % self.n * self.step, self.step)

    def blocks(self):
        """All of them, in one cut."""
        return self.panel.chunk(self.n, self.axis) if self.step else list(self)


class _Grid:
    """_shards without the R * C views: ``grid[i]`` is mesh row i's shards, ``_column(grid, j)`` mesh column j's."""

    def __init__(self, G: torch.Tensor, R: int, C: int):
        if G.dim() != 2:
            raise ValueError("operands must be 2-D")
        h, w = G.shape
        if h % R or w % C:
            raise ValueError(f"matrix {tuple(G.shape)} does not shard evenly over a {R}x{C} mesh")
        self.G, self.R, self.C, self.h, self.w = G, R, C, h // R, w // C

    def __len__(self):
        return self.R

    def __getitem__(self, i):
        if not -self.R <= i < self.R:
            raise IndexError(i)
        return _Line(self.G.narrow(0, i % self.R * self.h, self.h), self.C, 1, self.w)


def _row(grid, i, C):
    return grid[i] if isinstance(grid, _Grid) else [grid[i][j] for j in range(C)]


def _column(grid, j, R):
    return _Line(grid.G.narrow(1, j * grid.w, grid.w), R, 0, grid.h) if isinstance(grid, _Grid) else [grid[i][j] for i in range(R)]


def _shard(grid, i, j):
    return grid.G.narrow(0, i * grid.h, grid.h).narrow(1, j * grid.w, grid.w) if isinstance(grid, _Grid) else grid[i][j]


def _blocks(parts) -> Sequence[torch.Tensor]:
    """The shards of a mesh line as views, for a body that takes each of them more than once (a view per access to them made the overlapped bodies of
    2x2 devices in eight slices 7 % longer)."""
    return parts.blocks() if isinstance(parts, _Line) else parts


def _need(v: int, d: int, what: str) -> None:
    if d <= 0 or v % d:
        raise ValueError(f"{what} = {v} is not a multiple of {d}")


def _aligned(block: torch.Tensor) -> bool:
    """Whether a matrix's first element and its rows are 16-byte aligned."""
    return block.stride(1) == 1 and block.data_ptr() % 16 == 0 and (block.stride(0) * block.element_size()) % 16 == 0


def _own(block: torch.Tensor) -> torch.Tensor:
    """A device's shard as the kernels can address it: the view itself when it is aligned (a real device's shard is its own
    buffer), else a contiguous copy."""
    return block if _aligned(block) else block.contiguous()


def _gather(parts: Sequence[torch.Tensor], axis: int) -> torch.Tensor:
    """tiled all_gather of whole shards as the receiving device sees it: peers' parts concatenated in axis
    order, materialised contiguous in HBM (what a real all-gather delivers)."""
    return torch.cat(tuple(_blocks(parts)), dim=axis).contiguous()


PANEL_MAX_ROWS = 65535 * 8      # rows that one launch of the layout kernels always takes


def _spanning(parts: Sequence[torch.Tensor], axis: int):
    """The one view that covers ``parts`` when they are neighbouring blocks of one matrix in axis order (the shards of a
    global operand are), else None."""
    if isinstance(parts, _Line):
        p = parts.panel      # (rows that overlap, a window slid over a buffer, are rows of the shards only)
        return p if parts.axis == axis and p.stride(1) == 1 and p.shape[0] <= PANEL_MAX_ROWS and (axis == 0 or p.stride(0) >= p.shape[1]) else None
    p0 = parts[0]
    if len(parts) == 1:
        return p0 if p0.stride(1) == 1 and p0.shape[0] <= PANEL_MAX_ROWS else None
    step = p0.shape[1] if axis == 1 else p0.shape[0] * p0.stride(0)
    at, base = p0.storage_offset(), p0.untyped_storage().data_ptr()
    if p0.stride(1) != 1 or (axis == 1 and p0.stride(0) < len(parts) * p0.shape[1]):
        return None
    for p in parts:
        if (p.shape != p0.shape or p.stride() != p0.stride() or p.dtype != p0.dtype or p.device != p0.device
                or p.storage_offset() != at or p.untyped_storage().data_ptr() != base):
            return None
        at += step
    r, c = p0.shape
    if r * (1 if axis == 1 else len(parts)) > PANEL_MAX_ROWS:
        return None
    return p0.as_strided((r, c * len(parts)) if axis == 1 else (r * len(parts), c), p0.stride(), p0.storage_offset())


def _gather_col_slices(peers: Sequence[torch.Tensor], K: int, B: int) -> List[torch.Tensor]:
    """The K gathered column slices ``[rows, len(peers) * cols / K]``: every peer cuts its shard's columns into
    K block-cyclic slices (reference :155,157,198-199) and slice k of peer p lands at column block p of
    gathered slice k (all_gather over the peers' axis, tiled along the columns).  One kernel per peer writes
    its K slices straight into their places; there is no separate concatenation.  A shard is a whole number of rounds of
    K blocks, so peers that lie side by side in one matrix are cut by one kernel: the block-cyclic slices of the whole
    are the peers' slices side by side (the LS body of one device of a 2x4 mesh, 4096 x 4096 x 8192 in eight slices,
    128 -> 72 us, cheaper calls included)."""
    r, c = peers[0].shape
    _need(c, K * B, "sliced extent")
    w = c // K
    panel = _spanning(peers, 1)
    if panel is not None:
        return slice_layout.pack_slices(panel, K, B, 1)
    buf = torch.empty((K, r, len(peers) * w), dtype=peers[0].dtype, device=peers[0].device)
    for p, blk in enumerate(peers):
        slice_layout.pack_slices(blk, K, B, 1, out=[buf[k][:, p * w:(p + 1) * w] for k in range(K)])
    return [buf[k] for k in range(K)]


def _gather_row_slices(peers: Sequence[torch.Tensor], K: int, B: int) -> List[torch.Tensor]:
    """The K gathered row slices ``[len(peers) * rows / K, cols]`` (reference :156,158,177-178), peer p's part
    of slice k at row block p; one kernel for peers that lie one above the other in one matrix, else one per peer."""
    r, c = peers[0].shape
    _need(r, K * B, "sliced extent")
    h = r // K
    panel = _spanning(peers, 0)
    if panel is not None:
        return slice_layout.pack_slices(panel, K, B, 0)
    buf = torch.empty((K, len(peers) * h, c), dtype=peers[0].dtype, device=peers[0].device)
    for p, blk in enumerate(peers):
        slice_layout.pack_slices(blk, K, B, 0, out=[buf[k][p * h:(p + 1) * h] for k in range(K)])
    return [buf[k] for k in range(K)]


def _steps_addressable(row_bytes: int, K: int) -> bool:
    """Whether a K step of a product whose contraction runs through K row slices in place (eight blocks of a slice's rows, 8 * K rows apart)
    stays within the kernels' 32-bit offsets: always, but for slices of a few rows of hundreds of megabytes."""
    return 64 * K * row_bytes <= 1 << 32


def _addressable(t: torch.Tensor, K: int = 0) -> bool:
    """Whether the kernels can read a matrix as it stands, with K row slices in place as the slices of a contraction."""
    rows, cols = t.shape
    ld, step = t.stride()
    row = ld * t.element_size()
    return step == 1 and t.data_ptr() % 16 == 0 and row % 16 == 0 and ld >= cols and rows * row < 1 << 31 and _steps_addressable(row, K)


def _readable(parts: Sequence[torch.Tensor], axis: int):
    """_spanning's view where it is addressable, else None."""
    whole = _spanning(parts, axis)
    return whole if whole is not None and _addressable(whole) else None


def _gathered(parts: Sequence[torch.Tensor], axis: int) -> torch.Tensor:
    """_gather's matrix; shards that lie side by side in one matrix are that already and are not copied."""
    whole = _readable(parts, axis)
    return _gather(parts, axis) if whole is None else whole


def _uncut(peers: Sequence[torch.Tensor], K: int, B: int):
    """The gathered rows of which _gather_row_slices makes slices, where the kernels can read the slices inside them (blocks of eight rows
    of one matrix), else None.  The peers' slices one below the other are the slices of the whole, as in _gather_col_slices; the copy
    was 9 of 44 us of the LS body of one device of a 2x4 mesh, 4096 x 4096 x 8192 in eight slices."""
    _need(peers[0].shape[0], K * B, "sliced extent")
    return _readable(peers, 0) if B == 8 and K > 1 else None


# ------------------------------------------------------------------------------------------------
# per-device bodies.  X, W are the shard grids; (i, j) the device; the return value is what that
# device holds after its local contractions.
# ------------------------------------------------------------------------------------------------

def Collective_OS(X, W, i, j, R, C, K, B):
    """reference TensorParallel.py:19-22: gather X over col, W over row, one contraction."""
    Xi = _gathered(_row(X, i, C), 1)
    Wj = _gathered(_column(W, j, R), 0)
    return local_gemm.gemm_os([Xi], [Wj])


def Collective_LS(X, W, i, j, R, C, K, B):
    """reference :24-27: gather W over row; partial product X_ij @ Wj^T (input of psum_scatter)."""
    Wj = _gathered(_column(W, j, R), 0)
    return local_gemm.gemm_ls(_own(_shard(X, i, j)), [Wj])


def Collective_RS(X, W, i, j, R, C, K, B):
    """reference :29-32: gather X over col; partial product Xi^T @ W_ij (input of psum_scatter)."""
    Xi = _gathered(_row(X, i, C), 1)
    return local_gemm.gemm_rs([Xi], _own(_shard(W, i, j)))


def MeshFlow_OS(X, W, i, j, R, C, K, B):
    """reference :153-172: K gathered slice pairs, accumulated into one output block."""
    if K == 1:
        raise ValueError("the sliced OS body is undefined for K == 1 (the reference adds slice 0 twice); "
                         "use algorithm='collective' for the unsliced product")
    A_slices, peers = _gather_col_slices(_row(X, i, C), K, B), _column(W, j, R)
    W_rows = _uncut(peers, K, B)
    if W_rows is not None and _addressable(W_rows, K):
        return local_gemm.gemm_os_cyclic(A_slices, W_rows)
    return local_gemm.gemm_os(A_slices, _gather_row_slices(peers, K, B))


_gather_streams = {}           # (device, handle of the product's stream) -> the stream for its gathers, or None
_gather_streams_lock = threading.Lock()
_GATHER_STREAMS_MAX = 16
_GATHER_STREAM_TRIES = 6
_PROBE_TIMEOUT_MS = 50
OVERLAP_RESERVED_CUS = 32      # compute units left to the emulated gathers' copy kernels beside the waiting product


def _col_slice_filler(peers, K, B):
    """(buffer ``[K, rows, len(peers) * cols / K]`` for the K gathered column slices, ``fill(k)`` that gathers slice k into
    it on the current stream): slice k of a shard is its B-wide column blocks b with b % K == k (reference :155,157,198-199)."""
    peers = _blocks(peers)
    r, c = peers[0].shape
    _need(c, K * B, "sliced extent")
    w = c // K
    buf = torch.empty((K, r, len(peers) * w), dtype=peers[0].dtype, device=peers[0].device)

    def fill(k):
        for p, blk in enumerate(peers):
            buf[k][:, p * w:(p + 1) * w].copy_(blk.reshape(r, w // B, K, B)[:, :, k, :].reshape(r, w))
    return buf, fill


def _row_slice_filler(peers, K, B):
    """The same for the K gathered row slices ``[K, len(peers) * rows / K, cols]`` (reference :156,158,177-178)."""
    peers = _blocks(peers)
    h, n = peers[0].shape
    _need(h, K * B, "sliced extent")
    hk = h // K
    buf = torch.empty((K, len(peers) * hk, n), dtype=peers[0].dtype, device=peers[0].device)

    def fill(k):
        for p, blk in enumerate(peers):
            buf[k][p * hk:(p + 1) * hk].copy_(blk.reshape(hk // B, K, B, n)[:, k].reshape(hk, n))
    return buf, fill


def _runs_beside(cur, other, dev) -> bool:
    """Whether kernels on stream ``other`` run while a launch on ``cur`` waits.  The streams of a process share a few
    hardware queues and two that share one run in order, so the device is asked: the smallest gated product waits, at
    most _PROBE_TIMEOUT_MS, for a flag that ``other`` raises."""
    ready = torch.zeros(2, dtype=torch.int32, device=dev)
    a = torch.zeros((8, 512), dtype=torch.bfloat16, device=dev)
    b = torch.zeros((512, 8), dtype=torch.bfloat16, device=dev)
    other.wait_stream(cur)
    local_gemm.gemm_os_gated([a], [b], ready, timeout_ms=_PROBE_TIMEOUT_MS)
    with torch.cuda.stream(other):
        local_gemm.signal_set(ready, 0)
    cur.wait_stream(other)
    return not local_gemm.gate_timed_out(ready)


def _gather_stream(dev, cur):
    """The stream on which the gathers of an overlapped body on stream ``cur`` run: one that has been seen to run beside a
    waiting launch there, or None if none of a few does.  Looked for once per stream (the first call waits for the device
    to go idle, so that the search measures queues and not what stands in them)."""
    key = (dev, cur.cuda_stream)
    with _gather_streams_lock:
        if key in _gather_streams:
            return _gather_streams[key]
    torch.cuda.synchronize(dev)
    found = None
    for _ in range(_GATHER_STREAM_TRIES):
        stream = torch.cuda.Stream(dev)
        if _runs_beside(cur, stream, dev):
            found = stream
            break
    with _gather_streams_lock:
        _gather_streams[key] = found
        while len(_gather_streams) > _GATHER_STREAMS_MAX:
            del _gather_streams[next(iter(_gather_streams))]
    return found


def _launch_beside_reserved_units(launch, ready):
    lib = local_gemm._lib.load()
    try:
        lib.ms_set_reserved_cus(OVERLAP_RESERVED_CUS)
        return launch(ready)
    finally:
        lib.ms_set_reserved_cus(0)


def _fill_and_flag(K, ready, fills):
    for k in range(K):
        for fill in fills:
            fill(k)
        local_gemm.signal_set(ready, k)


def _launch_ahead_of_gathers(K, dev, launch, fills):
    """``launch(ready)`` enqueues the gated product on the current stream with all K flags down; the emulated gather
    stream then fills slice after slice (``fills``: one callable per gathered operand) and raises its flag.  On a real
    mesh that stream is the collective's.  Where no stream runs beside the waiting product the gathers go first; where
    they came too late for its time limit all the same (a stream that has been given another hardware queue since, a busy
    device), the product runs again on the slices that have arrived by then."""
    ready = torch.zeros(K + 1, dtype=torch.int32, device=dev)
    cur = torch.cuda.current_stream(dev)
    gather = _gather_stream(dev, cur)
    if gather is None:
        _fill_and_flag(K, ready, fills)
        return _launch_beside_reserved_units(launch, ready)
    gather.wait_stream(cur)                              # the flags are cleared and the shards are there
    out = _launch_beside_reserved_units(launch, ready)
    try:
        with torch.cuda.stream(gather):
            _fill_and_flag(K, ready, fills)
    finally:
        cur.wait_stream(gather)
    if local_gemm.gate_timed_out(ready):
        with _gather_streams_lock:
            _gather_streams.pop((dev, cur.cuda_stream), None)
        ready[K:].zero_()
        out = _launch_beside_reserved_units(launch, ready)
    return out


def MeshFlow_OS_overlap(X, W, i, j, R, C, K, B):
    """MeshFlow_OS in the order the reference's schedule runs it (:163-171): the product is launched once, before any
    slice has arrived, and multiplies slice k while the gathers of the later slices are still under way
    (``gemm_os_gated``).  The emulated gather stream fills slice k of both operands, peer by peer, and raises flag k.
    Same result as MeshFlow_OS on the compute units left to it, bit for bit, where that is one launch split the same way (a
    gated product is never done in two)."""
    if K == 1:
        raise ValueError("the sliced OS body is undefined for K == 1 (the reference adds slice 0 twice); "
                         "use algorithm='collective' for the unsliced product")
    bufA, fillA = _col_slice_filler(_row(X, i, C), K, B)
    bufB, fillB = _row_slice_filler(_column(W, j, R), K, B)
    return _launch_ahead_of_gathers(K, bufA.device, lambda ready: local_gemm.gemm_os_gated([bufA[k] for k in range(K)], [bufB[k] for k in range(K)], ready),
                                    (fillA, fillB))


def MeshFlow_LS_overlap(X, W, i, j, R, C, K, B):
    """MeshFlow_LS with the one launch ahead of the gathers of W's row slices (:176-189; ``gemm_ls_gated``): chunk k is
    multiplied as soon as slice k has arrived.  Same chunks as MeshFlow_LS, bit for bit."""
    bufW, fillW = _row_slice_filler(_column(W, j, R), K, B)
    own = _own(_shard(X, i, j))
    return _launch_ahead_of_gathers(K, bufW.device, lambda ready: local_gemm.gemm_ls_gated(own, [bufW[k] for k in range(K)], ready), (fillW,))


def MeshFlow_RS_overlap(X, W, i, j, R, C, K, B):
    """MeshFlow_RS with the one launch ahead of the gathers of X's column slices (:198-212; ``gemm_rs_gated``)."""
    bufX, fillX = _col_slice_filler(_row(X, i, C), K, B)
    own = _own(_shard(W, i, j))
    return _launch_ahead_of_gathers(K, bufX.device, lambda ready: local_gemm.gemm_rs_gated([bufX[k] for k in range(K)], own, ready), (fillX,))


def MeshFlow_LS(X, W, i, j, R, C, K, B):
    """reference :174-193: K gathered row slices of W; K fp32 partial chunks X_ij @ W_k^T."""
    own, peers = _own(_shard(X, i, j)), _column(W, j, R)
    W_rows = _uncut(peers, K, B)
    if W_rows is not None:
        return local_gemm.gemm_ls_cyclic(own, W_rows, K)
    return local_gemm.gemm_ls(own, _gather_row_slices(peers, K, B))


def MeshFlow_RS(X, W, i, j, R, C, K, B):
    """reference :195-214: K gathered column slices of X; K fp32 partial chunks X_k^T @ W_ij."""
    X_slices = _gather_col_slices(_row(X, i, C), K, B)
    return local_gemm.gemm_rs(X_slices, _own(_shard(W, i, j)))


# ------------------------------------------------------------------------------------------------
# ring baselines.  In the reference the halves of one operand (or of the partial output) travel round a
# mesh axis with ppermute, one hop per step, and each step multiplies two half-blocks (Wang_OS/LS/RS,
# reference :34-149; Cannon_OS/LS/RS, :218-342).  Seen from one device that is the same local
# contraction as the unsliced body, cut into 2 * size half-blocks taken in the order of their arrival:
# one kernel call with 2 * size slices (OS) or 2 * size chunks written to their places in the device's
# partial output (LS / RS).  The reference reads the device's ring position with ``jax.lax.ax_index``,
# a name JAX does not have; the position is taken here as ``axis_index`` gives it.
# ------------------------------------------------------------------------------------------------

def _ring_order(algorithm: str, dataflow: str, R: int, C: int, i: int, j: int):
    """[(block, half)] in step order for device (i, j).  Wang: ring = the mesh row; the low halves come from
    the left (block j, j-1, ..), the high halves from the right (j, j+1, ..); for LS the partial outputs
    travel instead and a device works on block j-1-t / j+1+t in step t (reference :45-59, :76-89,
    :132-146).  Cannon (square mesh): both start at k = (i + j) % N, low halves move on to k+1, k+2, ..,
    high halves to k-1, k-2, .. (:235-259, :268-294, :309-335)."""
    if algorithm == "wang":
        if dataflow == "ls":
            return [p for t in range(C) for p in (((j - 1 - t) % C, 0), ((j + 1 + t) % C, 1))]
        return [p for t in range(C) for p in (((j - t) % C, 0), ((j + t) % C, 1))]
    k = (i + j) % C
    return [p for t in range(C) for p in (((k + t) % C, 0), ((k - t) % C, 1))]


def _usable(views: Sequence[torch.Tensor]) -> List[torch.Tensor]:
    """The views themselves if the kernels can address all of them in place, else contiguous copies of all
    (slices of one call share a leading dimension)."""
    if all(_aligned(v) for v in views):
        return list(views)
    return [v.contiguous() for v in views]


def _halves(parts, axis: int) -> Sequence[torch.Tensor]:
    """The half-blocks of a mesh line's shards, cut across ``axis``: half ``hi`` of block ``b`` is number ``2 * b + hi``.  (One cut of the view
    that covers the line: a view per access to its shards took one device of 2 x 4 some 20 us of the host.)"""
    width = parts.step if isinstance(parts, _Line) else parts[0].shape[axis]
    _need(width, 2, "sliced extent of a shard")
    return _cut(parts.panel, width // 2, axis) if isinstance(parts, _Line) else [v for p in parts for v in _cut(p, width // 2, axis)]


def _cut(t: torch.Tensor, h: int, axis: int) -> Sequence[torch.Tensor]:
    if h < 1:
        raise ValueError(f"matrix {tuple(t.shape)} has no half-blocks")
    return t.chunk(t.shape[axis] // h, axis)


def _ring_os(algorithm, X, W, i, j, R, C):
    Wj = _gathered(_column(W, j, R), 0)                     # [Kd, n/C]
    halves = _halves(_row(X, i, C), 1)
    _need(Wj.shape[0], 2 * C, "gathered rows of W")
    order = [2 * b + hi for b, hi in _ring_order(algorithm, "os", R, C, i, j)]
    rows = _cut(Wj, Wj.shape[0] // C // 2, 0)
    return local_gemm.gemm_os(_usable([halves[x] for x in order]), [rows[x] for x in order])


def _ring_ls(algorithm, X, W, i, j, R, C):
    Wj = _gathered(_column(W, j, R), 0)                     # [O, I/C]
    _need(Wj.shape[0], 2 * C, "gathered rows of W")
    h = Wj.shape[0] // C // 2
    order = [2 * b + hi for b, hi in _ring_order(algorithm, "ls", R, C, i, j)]
    Xij = _own(_shard(X, i, j))
    part = torch.empty((Xij.shape[0], Wj.shape[0]), dtype=torch.float32, device=Xij.device)
    rows, columns = _cut(Wj, h, 0), _cut(part, h, 1)
    if any(columns[x].data_ptr() % 16 for x in order):
        raise ValueError(f"half-blocks of {h} output columns are not 16-byte aligned")
    local_gemm.gemm_ls(Xij, [rows[x] for x in order], out=[columns[x] for x in order])
    return [part]


def _ring_rs(algorithm, X, W, i, j, R, C):
    halves = _halves(_row(X, i, C), 1)
    h = halves[0].shape[1]
    order = [2 * b + hi for b, hi in _ring_order(algorithm, "rs", R, C, i, j)]
    Xs = _usable([halves[x] for x in order])
    Wij = _own(_shard(W, i, j))
    part = torch.empty((2 * h * C, Wij.shape[1]), dtype=torch.float32, device=Wij.device)
    rows = _cut(part, h, 0)
    local_gemm.gemm_rs(Xs, Wij, out=[rows[x] for x in order])
    return [part]


def Wang_OS(X, W, i, j, R, C, K, B):
    """reference :34-61."""
    return _ring_os("wang", X, W, i, j, R, C)


def Wang_LS(X, W, i, j, R, C, K, B):
    """reference :64-90; returns the device's whole partial output ``X_ij @ Wj^T`` (what the travelling
    half-blocks sum up over the mesh row)."""
    return _ring_ls("wang", X, W, i, j, R, C)


def Wang_RS(X, W, i, j, R, C, K, B):
    """reference :92-149 (the branch it takes, :120-149); returns the device's partial ``Xi^T @ W_ij``."""
    return _ring_rs("wang", X, W, i, j, R, C)


def Cannon_OS(X, W, i, j, R, C, K, B):
    """reference :218-260."""
    return _ring_os("cannon", X, W, i, j, R, C)


def Cannon_LS(X, W, i, j, R, C, K, B):
    """reference :262-300."""
    return _ring_ls("cannon", X, W, i, j, R, C)


def Cannon_RS(X, W, i, j, R, C, K, B):
    """reference :379-417 (the definition in force: it shadows the one at :302-342, which computes the same product)."""
    return _ring_rs("cannon", X, W, i, j, R, C)


# ------------------------------------------------------------------------------------------------
# mesh completion: what psum_scatter + the (.., K, B) interleave do with the partial chunks
# ------------------------------------------------------------------------------------------------

def _block(extent: int, B: int) -> int:
    """Largest block size <= B (a power of two) in which ``extent`` divides: the unsliced bodies have no block size of
    their own, and a window of any width is a whole number of blocks of 1."""
    while B > 1 and extent % B:
        B //= 2
    return max(B, 1)


def _finish(chunks_by_peer, me, axis, B, dtype):
    """psum_scatter over the peers (device ``me`` of them keeps its window of every summed chunk) and the
    interleave of the K windows into the output shard: reference :182-193 (LS: peers = the mesh row,
    axis 1) and :204-214 (RS: peers = the mesh column, axis 0); with one chunk per peer it is the tiled scatter of
    the unsliced bodies (:27, :32).  One layout kernel; the sum is fp32 in peer order with one rounding to ``dtype``.
    More than 64 chunk pointers (P * K) do not fit one launch: the peers are then summed group by group into fp32
    shards, and one more launch adds those up and rounds."""
    P, K = len(chunks_by_peer), len(chunks_by_peer[0])
    if P * K <= 64:
        return slice_layout.unpack_chunks(chunks_by_peer, B, axis, window=me, parts=P, out_dtype=dtype)
    g = max(1, 64 // K)
    partial = [slice_layout.unpack_chunks(chunks_by_peer[p0:p0 + g], B, axis, window=me, parts=P, out_dtype=torch.float32)
               for p0 in range(0, P, g)]
    width = partial[0].shape[1] if axis == 1 else partial[0].shape[0]
    return slice_layout.unpack_chunks([[t] for t in partial], _block(width, 8), axis, window=0, parts=1, out_dtype=dtype)


# ------------------------------------------------------------------------------------------------
# the whole mesh at once.  On the one GPU that plays every device, the devices of a mesh row or column receive the same
# gathered slices, and their products differ only in which rows and columns of them they take: one kernel gathers an operand
# for all of them (see _spanning), one product covers them all.  Device by device a training step of a small layer is some
# 150 launches of 2 to 40 us, bound by the host that issues them: 512 x 256 x 1024 on a 4x2 mesh 3.7 ms, in this way 0.40;
# 2048 x 3072 x 12288 on a 2x4 mesh 5.1 ms, in this way 0.56.  The price is memory: gathered operands and partial chunks of
# all mesh lines are alive at once, where device by device it is one line's.  bf16 products of LS and RS need neither (_sums_on_chip):
# their sums over a mesh line stay in registers, and the two training steps take 0.23 and 0.43 ms.
# ------------------------------------------------------------------------------------------------

WHOLE_MESH_MAX_CHUNK_BYTES = 4 << 30      # partial chunks alive at once; device by device it is one mesh line's


def _fits_whole_mesh(dataflow, X, W, R, C, K) -> bool:
    """Whether the mesh's products can run as one: every device's own extents are ones that the kernels take (a mesh whose
    devices would be refused is refused), no operand reaches the 2 GiB that a kernel addresses, the line's chunks fit one
    pointer table (64) and a bounded buffer, and rows fit one launch of the layout kernels.  (Whether it all fits the memory
    that is left shows when it is allocated, see ShardedMatmul.__call__.)"""
    q = 16 // X.element_size()
    if X.device != W.device or X.dtype not in (torch.float32, torch.bfloat16) or X.stride(1) != 1 or W.stride(1) != 1:
        return False
    if max(X.shape[0], W.shape[0]) > PANEL_MAX_ROWS or min(X.numel(), W.numel()) == 0:
        return False
    if any(t.shape[0] * max(t.stride(0), t.shape[1]) * t.element_size() >= 1 << 31 for t in (X, W)):
        return False
    if dataflow == "os":
        return (W.shape[1] // C) % q == 0 and (X.shape[1] // K) % q == 0 and K <= 64
    if dataflow == "ls":
        peers, m, n, aligned = C, X.shape[0], W.shape[0], (X.shape[1] // C, W.shape[0] // K, W.shape[0] // C)
    else:
        peers, m, n, aligned = R, X.shape[1], W.shape[1], (W.shape[1] // C, X.shape[1] // K, W.shape[1])
    return peers * K <= 64 and peers * m * n * 4 <= WHOLE_MESH_MAX_CHUNK_BYTES and m <= PANEL_MAX_ROWS and not any(v % q for v in aligned)


def _whole_os(X, W, K, B):
    """The output blocks of all devices are one product, whose gathered slices hold every device's."""
    return local_gemm.gemm_os(slice_layout.pack_slices(X, K, B, 1), slice_layout.pack_slices(W, K, B, 0))


def _whole_ls(X, W, C, K, B, sliced):
    """Every device's partial chunks in one launch and their reduce-scatters in another: mesh column j multiplies its columns
    of X (the rows of all mesh rows together) with its columns of the gathered slices of W; the sum over j is fp32 in peer
    order, as in _finish, and the windows of all devices together are the whole chunks."""
    slices = slice_layout.pack_slices(W, K, B, 0) if sliced else [_gather([W], 0)]
    w = X.shape[1] // C
    A = _usable([X[:, j * w:(j + 1) * w] for j in range(C)])
    chunks = local_gemm.gemm_ls_peers(A, [[t[:, j * w:(j + 1) * w] for t in slices] for j in range(C)])
    return slice_layout.unpack_chunks(chunks, B if sliced else _block(W.shape[0], 8), 1, out_dtype=X.dtype)


def _whole_rs(X, W, R, K, B, sliced):
    """The same for the right-hand-stationary dataflow: mesh row i multiplies its rows of the gathered slices of X with its
    rows of W."""
    slices = slice_layout.pack_slices(X, K, B, 1) if sliced else [_gather([X], 1)]
    h = X.shape[0] // R
    own = _usable([W[i * h:(i + 1) * h] for i in range(R)])
    chunks = local_gemm.gemm_rs_peers([[t[i * h:(i + 1) * h] for t in slices] for i in range(R)], own)
    return slice_layout.unpack_chunks(chunks, B if sliced else _block(X.shape[1], 8), 0, out_dtype=X.dtype)


def _sums_on_chip(X, W) -> bool:
    """Whether a line's partial sums can be added up inside the product (local_gemm.gemm_ls_sum, gemm_rs_sum) instead of as fp32 chunks
    in memory: bf16 operands that the kernel can address in place.  That writes a tenth of the bytes: LS 2048 x 3072 x 12288 of four devices
    172 -> 128 us, RS 3072 x 12288 x 2048 of two 251 -> 131, small ones a quarter of the launches (512 x 256 x 1024 on 4x2 97 -> 23 us).
    Where the contraction is long it can be the slower way: local_gemm.prefers_sum prices both."""
    if X.dtype != torch.bfloat16:
        return False
    x, w = X.stride(0), W.stride(0)
    return (X.data_ptr() | W.data_ptr()) % 16 == 0 and (x | w) % 8 == 0 and x >= X.shape[1] and w >= W.shape[1]


def _half_blocks_fit(dataflow, X, W, C) -> bool:
    """Whether the ring bodies of every device take these operands, and the kernels can address them: half-blocks that are whole pieces of 16
    bytes, rows that do not overlap (others are refused, or copied, device by device)."""
    q = 16 // X.element_size()
    extent = W.shape[0] if dataflow == "ls" else X.shape[1]
    return extent % (2 * C * q) == 0 and C <= 32 and X.stride(0) >= X.shape[1] and W.stride(0) >= W.shape[1]


# Bytes of a column's output block from which it is worth 15 us more of the host (a call with ``out=`` is not native) to have it written where it belongs
# instead of copied there.  2x2 devices, 2048 x 2048 x 2048 69 us with out=, 39 without, 4096 x 4096 x 1024 (32 MB) 69 and 63, 8192 x 8192 x 1024 114 and 212; 1x4, 4096 x 12288 x 512
# (96 MB) 174 and 138, 8192 x 8192 x 1024 (128 MB) 172 and 225.
RING_IN_PLACE_BYTES = 20 << 20


def _whole_ring_os(X, W, C):
    """The devices of a mesh column add up the same half-blocks in the same order, so their output blocks are one product: C of them instead of R * C.
    (The chunks of the ring LS and RS bodies are Collective's partial sums, cut in two.)"""
    h, n = X.shape[1] // C // 2, W.shape[1] // C
    halves, columns = X.split(h, 1), W.split(n, 1)
    Y = None
    if C > 1 and X.shape[0] * n * X.element_size() > RING_IN_PLACE_BYTES:
        Y = torch.empty((X.shape[0], W.shape[1]), dtype=X.dtype, device=X.device)
    blocks = []
    for j in range(C):
        order = [2 * b + hi for b, hi in _ring_order("wang", "os", 1, C, 0, j)]
        rows = columns[j].split(h, 0)
        blocks.append(local_gemm.gemm_os(_usable([halves[x] for x in order]), _usable([rows[x] for x in order]), out=None if Y is None else Y[:, j * n:(j + 1) * n]))
    return Y if Y is not None else torch.cat(blocks, 1) if C > 1 else blocks[0]


# (the bodies launched ahead of their gathers keep a product per device where that produces chunks; of the ring bodies only Cannon's OS, whose devices
# in step with each other make no rectangle)
_RING_BODIES = (Wang_OS, Wang_LS, Wang_RS, Cannon_LS, Cannon_RS)
_WHOLE_MESH_BODIES = {"os": (Collective_OS, MeshFlow_OS, MeshFlow_OS_overlap, Wang_OS), "ls": (Collective_LS, MeshFlow_LS, Wang_LS, Cannon_LS),
                      "rs": (Collective_RS, MeshFlow_RS, Wang_RS, Cannon_RS)}


class ShardedMatmul:
    """What ``SPMD.OS/LS/RS(K)`` returns: ``f(X, W) -> Y`` on global operands, plus ``f.device(i, j)``."""

    def __init__(self, dataflow: str, body: Callable, mesh: Mesh, K: int, B: int, sliced: bool):
        self.dataflow, self.body, self.mesh, self.K, self.B, self.sliced = dataflow, body, mesh, int(K), int(B), sliced
        self.R, self.C = mesh.shape

    # shape rules implied by the reference's reshapes (:155-156,177-179,198-200)
    def _validate(self, X: torch.Tensor, W: torch.Tensor) -> None:
        R, C = self.R, self.C
        S = self.K if self.sliced else 1
        B = self.B if self.sliced else 1
        if S < 1:
            raise ValueError(f"slice count must be >= 1, got {S}")
        for t, name in ((X, "X"), (W, "W")):
            if not isinstance(t, torch.Tensor) or t.dim() != 2:
                raise ValueError(f"{name} must be a 2-D torch tensor")
        if X.dtype != W.dtype:
            raise ValueError("X and W must share a dtype")
        if self.dataflow == "os":
            if X.shape[1] != W.shape[0]:
                raise ValueError(f"os: cannot contract {tuple(X.shape)} @ {tuple(W.shape)}")
            _need(X.shape[0], R, "rows of X"); _need(W.shape[1], C, "cols of W")
            _need(X.shape[1], C * S * B, "cols of X"); _need(W.shape[0], R * S * B, "rows of W")
        elif self.dataflow == "ls":
            if X.shape[1] != W.shape[1]:
                raise ValueError(f"ls: cannot contract {tuple(X.shape)} @ {tuple(W.shape)}^T")
            _need(X.shape[0], R, "rows of X"); _need(X.shape[1], C, "cols of X")
            _need(W.shape[0], R * S * B, "rows of W"); _need(W.shape[0], C * S * B, "rows of W")
        else:
            if X.shape[0] != W.shape[0]:
                raise ValueError(f"rs: cannot contract {tuple(X.shape)}^T @ {tuple(W.shape)}")
            _need(X.shape[0], R, "rows of X"); _need(W.shape[1], C, "cols of W")
            _need(X.shape[1], C * S * B, "cols of X"); _need(X.shape[1], R * S * B, "cols of X")
        for t, name in ((X, "X"), (W, "W")):
            if not t.is_cuda:
                raise local_gemm._lib.MeshSliceError(f"{name} must live on the GPU: there is no CPU path")

    def device(self, i: int, j: int) -> Callable:
        """Body of mesh device (i, j): returns its output block (OS) or its fp32 partial chunks."""
        if not (0 <= i < self.R and 0 <= j < self.C):
            raise ValueError(f"device ({i},{j}) is outside the {self.R}x{self.C} mesh")

        def run(X, W):
            self._validate(X, W)
            return self.body(_Grid(X, self.R, self.C), _Grid(W, self.R, self.C), i, j, self.R, self.C, self.K, self.B)
        return run

    def _whole_mesh(self, X, W, K, B):
        if self.body is Wang_OS:
            return _whole_ring_os(X, W, self.C)
        if self.dataflow == "os":      # (the other bodies: on a mesh of one)
            return _whole_os(X, W, K, B) if self.body is MeshFlow_OS and K > 1 else self.body([[X]], [[W]], 0, 0, 1, 1, self.K, self.B)
        return _whole_ls(X, W, self.C, K, B, self.sliced) if self.dataflow == "ls" else _whole_rs(X, W, self.R, K, B, self.sliced)

    def __call__(self, X: torch.Tensor, W: torch.Tensor) -> torch.Tensor:
        self._validate(X, W)
        R, C = self.R, self.C
        K = self.K if self.sliced else 1
        B = self.B if self.sliced else 1
        if (self.body in _WHOLE_MESH_BODIES[self.dataflow] and _fits_whole_mesh(self.dataflow, X, W, R, C, K)
                and (self.body not in _RING_BODIES or _half_blocks_fit(self.dataflow, X, W, C))):
            try:
                # (nothing that the kernels can read in place is gathered, cut or interleaved: an OS product's slices decide the order in which it
                # contracts, the sums over a line are the same whatever the slices)
                if self.body is MeshFlow_OS and K > 1 and B == 8 and _addressable(W, K):
                    return local_gemm.gemm_os_cyclic(slice_layout.pack_slices(X, K, B, 1), W)
                if self.dataflow == "ls" and _sums_on_chip(X, W):
                    m, k = X.shape
                    if local_gemm.prefers_sum("ls", C, K, m, W.shape[0], k // C):
                        return local_gemm.gemm_ls_sum(X, W, C)
                elif self.dataflow == "rs" and _sums_on_chip(X, W):
                    k, m = X.shape
                    if local_gemm.prefers_sum("rs", R, K, m, W.shape[1], k // R):
                        return local_gemm.gemm_rs_sum(X, W, R)
                return self._whole_mesh(X, W, K, B)
            except torch.OutOfMemoryError:
                pass       # what all mesh lines need at once (slices of all of X, gathered operands, chunks) does not fit beside the caller's tensors: one line's may
        Xs, Ws = _shards(X, R, C), _shards(W, R, C)
        run = lambda i, j: self.body(Xs, Ws, i, j, R, C, self.K, self.B)
        if self.dataflow == "os":
            return torch.cat([torch.cat([run(i, j) for j in range(C)], dim=1) for i in range(R)], dim=0)
        if self.dataflow == "ls":
            rows = []
            for i in range(R):
                chunks = [run(i, j) for j in range(C)]
                # (unsliced bodies bring one chunk each: the tiled scatter of contiguous column blocks)
                Bw = B if self.sliced else _block(chunks[0][0].shape[1] // C, 8)
                rows.append(torch.cat([_finish(chunks, j, 1, Bw, X.dtype) for j in range(C)], dim=1))
            return torch.cat(rows, dim=0)
        cols = []
        for j in range(C):
            chunks = [run(i, j) for i in range(R)]
            Bw = B if self.sliced else _block(chunks[0][0].shape[0] // R, 8)
            cols.append(torch.cat([_finish(chunks, i, 0, Bw, X.dtype) for i in range(R)], dim=0))
        return torch.cat(cols, dim=1)


class SPMD:
    """reference TensorParallel.py:346-377.  ``jit`` is accepted and ignored: kernels are ahead-of-time
    compiled."""

    def __init__(self, mesh: Mesh, algorithm: str = "collective", blocksize: int = 8, jit: bool = True):
        self.mesh = mesh
        self.rowaxis = mesh.axis_names[0]
        self.colaxis = mesh.axis_names[1]
        self.spec = P(self.rowaxis, self.colaxis)
        self.blocksize = blocksize
        self.jit = jit
        self.algorithm = algorithm
        if algorithm == "collective":
            self.funcs = {"os": Collective_OS, "ls": Collective_LS, "rs": Collective_RS}
            self.sliced = False
        elif algorithm == "wang":
            self.funcs = {"os": Wang_OS, "ls": Wang_LS, "rs": Wang_RS}
            self.sliced = False
        elif algorithm == "cannon":
            assert mesh.devices.shape[0] == mesh.devices.shape[1], "cannon needs a square mesh"
            self.funcs = {"os": Cannon_OS, "ls": Cannon_LS, "rs": Cannon_RS}
            self.sliced = False
        elif algorithm == "meshflow_overlap":      # MeshFlow with each device's one product launched ahead of its gathers
            self.funcs = {"os": MeshFlow_OS_overlap, "ls": MeshFlow_LS_overlap, "rs": MeshFlow_RS_overlap}
            self.sliced = True
        else:  # like the reference, any other name selects the sliced MeshFlow bodies
            self.funcs = {"os": MeshFlow_OS, "ls": MeshFlow_LS, "rs": MeshFlow_RS}
            self.sliced = True

    def _build(self, which: str, K: int) -> ShardedMatmul:
        if int(K) < 1:
            raise ValueError(f"slice count K must be >= 1, got {K}")
        return ShardedMatmul(which, self.funcs[which], self.mesh, K, self.blocksize, self.sliced)

    def OS(self, K: int = 8) -> ShardedMatmul:
        return self._build("os", K)

    def LS(self, K: int = 8) -> ShardedMatmul:
        return self._build("ls", K)

    def RS(self, K: int = 8) -> ShardedMatmul:
        return self._build("rs", K)


def createMultihostMatrix(mesh: Mesh, sharding, global_shape, dtype=torch.bfloat16, seed: int = 0, device="cuda"):
    """reference :419-423: a random N(0,1) matrix of ``global_shape`` sharded over the mesh.  The
    reference seeds JAX's generator with the process index; this build has one process and uses
    torch's generator with ``seed`` (the sample streams differ; nothing depends on them)."""
    g = torch.Generator(device="cpu").manual_seed(int(seed))
    return torch.randn(tuple(global_shape), generator=g, dtype=torch.float32).to(dtype).to(device)
