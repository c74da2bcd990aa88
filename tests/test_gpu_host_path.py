"""The native call path (csrc/ms_host.cpp) against the Python path that takes what it declines: same results, same refusals."""
import threading
import time

import pytest
import torch

import meshslice_amd as ms
from meshslice_amd import TensorParallel as TP, _lib, local_gemm
from meshslice_amd.slice_layout import pack_slices, unpack_chunks

pytestmark = pytest.mark.gpu


class _Declines:
    """The native path with every call declined (the workspace bookkeeping stays)."""

    def __getattr__(self, name):
        return getattr(_host, name) if name.startswith("workspace") else lambda *a: None


_host = _lib.host


def _calls(dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    A, B = [r(72, 40) for _ in range(3)], [r(40, 56) for _ in range(3)]
    wide, chunks = r(64, 96), [[r(32, 16).float() for _ in range(3)] for _ in range(2)]
    calls = [lambda: ms.gemm_os(A, B), lambda: ms.gemm_os(tuple(A), B, out_dtype=torch.float32), lambda: ms.gemm_ls(A[0], [a[:24] for a in A]),
             lambda: ms.gemm_ls(A[0], [A[1]], out_dtype=torch.bfloat16), lambda: ms.gemm_rs([a[:, :16] for a in A], A[2]),
             lambda: pack_slices(wide, 4, 8, 1), lambda: pack_slices(wide[:, 8:40], 2, 4, 0), lambda: pack_slices(wide[:, 1:41], 5, 8, 1),
             lambda: unpack_chunks(chunks, 8, 1, out_dtype=dtype), lambda: unpack_chunks(chunks, 8, 0, window=1, parts=2),
             lambda: local_gemm.gemm_os_cyclic([a[:, :32] for a in A[:2]], wide)]
    if dtype == torch.bfloat16:
        res = r(72, 64)[:, :56]
        calls += [lambda: ms.gemm_os(A, B, activation="gelu"), lambda: ms.gemm_os(A, B, residual=res), lambda: local_gemm.gemm_ls_sum(wide, wide, 3),
                  lambda: local_gemm.gemm_rs_sum(wide, wide, 2)]
    return calls


def _equal(a, b):
    if isinstance(a, torch.Tensor):
        return a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b) and not a.requires_grad
    return len(a) == len(b) and all(_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_both_paths_give_the_same(dtype, monkeypatch):
    calls = _calls(dtype, 1)
    ms.gemm_os(*[[torch.zeros(8, 8, device="cuda")]] * 2)      # (the stream's workspace)
    got = [f() for f in calls]
    other, side = torch.cuda.Stream(), []
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        side = [f() for f in calls]
    torch.cuda.synchronize()
    monkeypatch.setattr(_lib, "host", _Declines())
    want = [f() for f in calls]
    for i, (a, b, c) in enumerate(zip(got, want, side)):
        assert _equal(a, b) and _equal(c, b), i


def test_the_native_path_takes_the_ordinary_calls():
    """None of these goes through the Python path."""
    a = torch.randn(16, 16, device="cuda").bfloat16()
    ms.gemm_os([a], [a])
    h = _host
    for got in (h.gemm_os([a], [a], None, False, None), h.gemm_os((a, a), [a, a], torch.float32, True, a.float()), h.gemm_ls(a, [a], None), h.gemm_rs([a], a, None),
                h.gemm_ls_sum(a, a, 2), h.gemm_rs_sum(a, a, 2), h.gemm_os_cyclic([a[:, :8], a[:, 8:]], a), h.pack_slices(a, 2, 8, 1), h.unpack_chunks([[a], [a]], 8, 1, 0, 1, None)):
        assert got is not None


def test_what_the_native_path_declines():
    a = torch.randn(16, 16, device="cuda").bfloat16()
    ms.gemm_os([a], [a])
    h, odd = _host, torch.randn(16, 12, device="cuda").bfloat16()
    class Sub(torch.Tensor):
        pass
    declined = [h.gemm_os([a], [a, a], None, False, None), h.gemm_os([a.cpu()], [a], None, False, None), h.gemm_os([a.t()], [a], None, False, None),
                h.gemm_os([a], [a.float()], None, False, None), h.gemm_os([a], [a], torch.float16, False, None), h.gemm_os([], [], None, False, None),
                h.gemm_os([a] * 65, [a] * 65, None, False, None), h.gemm_os([odd], [odd.t().contiguous()], None, False, None), h.gemm_os(a, a, None, False, None),
                h.gemm_os([a.as_subclass(Sub)], [a], None, False, None), h.gemm_os([a], [a], None, False, odd), h.gemm_os([None], [a], None, False, None),
                h.gemm_os_cyclic([a], odd.t()), h.gemm_os_cyclic([a, a], a), h.gemm_ls(a, [odd], None), h.gemm_rs([a], None, None), h.gemm_ls_sum(a, a, 3), h.gemm_ls_sum(a, a, "2"), h.gemm_rs_sum(a.float(), a.float(), 2),
                h.pack_slices(a, 3, 8, 1), h.pack_slices(a, 0, 8, 1), h.pack_slices(a, 2, 8, 2), h.pack_slices(a, 2.0, 8, 1),
                h.unpack_chunks([[a], [a, a]], 8, 1, 0, 1, None), h.unpack_chunks([], 8, 1, 0, 1, None), h.unpack_chunks([[a]], 8, 1, 2, 2, None),
                h.unpack_chunks([[a] * 40, [a] * 40], 8, 1, 0, 1, None)]
    assert all(d is None for d in declined), [i for i, d in enumerate(declined) if d is not None]
    with torch.device("meta"):      # (a mode that the allocation would meet)
        assert h.gemm_os([a], [a], None, False, None) is None
    seen = []
    torch.func.vmap(lambda t: (seen.append(h.pack_slices(t, 2, 8, 1)), t)[1])(torch.stack([a, a]))
    assert seen == [None]
    with pytest.raises(ValueError):
        ms.gemm_os([a], [odd])
    with pytest.raises(TypeError):
        h.gemm_os([a])


def test_a_stream_under_capture_is_left_to_the_python_path():
    """Its workspace comes from the graph's own pool, and the graph's replays give the eager bits."""
    g = torch.Generator(device="cuda").manual_seed(3)
    A, B = [torch.randn(512, 2048, generator=g, device="cuda").bfloat16()], [torch.randn(2048, 512, generator=g, device="cuda").bfloat16()]
    want = ms.gemm_os(A, B)
    assert _lib.load().ms_query(_lib.MS_QUERY_LAST_SPLITS) > 1
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert _host.gemm_os(A, B, None, False, None) is None
        out = ms.gemm_os(A, B)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want) and torch.equal(ms.gemm_os(A, B), want)


def test_evicted_workspaces_are_not_handed_out_and_the_busiest_stays(monkeypatch):
    monkeypatch.setattr(local_gemm, "_WORKSPACE_CACHE_MAX", 3)
    a = torch.randn(16, 16, device="cuda").bfloat16()
    streams = [torch.cuda.Stream() for _ in range(5)]
    dev = torch.cuda.current_device()
    for s in streams:
        with torch.cuda.stream(s):
            ms.gemm_os([a], [a])
        with torch.cuda.stream(streams[0]):      # (taken from the native path's table each time)
            ms.gemm_os([a], [a])
    kept = {k[1] for k in local_gemm._workspaces if k[0] == dev}
    assert len(kept) <= 3 and streams[0].cuda_stream in kept
    for s in streams:
        assert bool(_host.workspace_touch(dev, s.cuda_stream, False)) == (s.cuda_stream in kept)
    torch.cuda.synchronize()


def test_threads_on_streams_of_their_own():
    g = torch.Generator(device="cuda").manual_seed(9)
    ops = [([torch.randn(256, 2048, generator=g, device="cuda").bfloat16()], [torch.randn(2048, 256, generator=g, device="cuda").bfloat16()]) for _ in range(4)]
    want = [ms.gemm_os(*o) for o in ops]
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                y = ms.gemm_os(*ops[i])
                torch.cuda.current_stream().synchronize()
                if not torch.equal(y, want[i]):
                    bad.append(i)
    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


@pytest.mark.parametrize("name", ["gemm_os", "gemm_ls", "pack_slices", "gemm_ls_sum"])
def test_a_call_that_waits_for_a_full_queue_does_not_stop_other_threads(name):
    """One thread queues calls behind a product that waits for its slice until the queue takes no more; the flag comes from another thread.
    The wait is bounded: a thread that could not run raises its flag too late, and the product says so."""
    dev, cur = torch.device("cuda", torch.cuda.current_device()), torch.cuda.current_stream()
    other = TP._gather_stream(dev, cur)
    if other is None:
        pytest.skip("no stream runs beside a waiting product")
    a, b = torch.randn(8, 512, device="cuda").bfloat16(), torch.randn(512, 8, device="cuda").bfloat16()
    call = {"gemm_os": lambda: ms.gemm_os([a], [b]), "gemm_ls": lambda: ms.gemm_ls(a, [a]), "pack_slices": lambda: pack_slices(a, 2, 8, 1),
            "gemm_ls_sum": lambda: local_gemm.gemm_ls_sum(a, a, 2)}[name]
    call()
    ready = torch.zeros(2, dtype=torch.int32, device="cuda")
    queued = []

    def fill():
        with torch.cuda.stream(cur):
            for i in range(40000):
                call()
                queued.append(i)
    torch.cuda.synchronize()
    local_gemm.gemm_os_gated([a], [b], ready, timeout_ms=4000)
    t = threading.Thread(target=fill)
    t.start()
    time.sleep(1.0)
    with torch.cuda.stream(other):
        local_gemm.signal_set(ready, 0)
    blocked = len(queued)
    t.join()
    torch.cuda.synchronize()
    assert not local_gemm.gate_timed_out(ready), f"{blocked} calls were queued"


def test_a_workspace_taken_away_during_a_call_lives_until_its_launch():
    """Evicted from the table while another thread's calls use it: no result changes and the counters it comes back with are zero."""
    g = torch.Generator(device="cuda").manual_seed(5)
    A, B = [torch.randn(256, 4096, generator=g, device="cuda").bfloat16()], [torch.randn(4096, 256, generator=g, device="cuda").bfloat16()]
    want = ms.gemm_os(A, B)
    assert _lib.load().ms_query(_lib.MS_QUERY_LAST_SPLITS) > 1
    stream, bad, stop = torch.cuda.Stream(), [], threading.Event()
    torch.cuda.synchronize()

    def work():
        with torch.cuda.stream(stream):
            for _ in range(400):
                y = ms.gemm_os(A, B)
                if not torch.equal(y, want):
                    bad.append(1)
        stop.set()
    t = threading.Thread(target=work)
    t.start()
    while not stop.is_set():
        for _ in range(12):      # (more streams than keep a workspace)
            with torch.cuda.stream(torch.cuda.Stream()):
                ms.gemm_os([A[0][:8]], B)
        time.sleep(0.001)
    t.join()
    torch.cuda.synchronize()
    assert not bad and len([k for k in local_gemm._workspaces if k[0] == torch.cuda.current_device()]) <= local_gemm._WORKSPACE_CACHE_MAX
    assert torch.equal(ms.gemm_os(A, B), want)
