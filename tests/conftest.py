import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")
    config.addinivalue_line("markers", "perf: asserts on wall-clock behaviour (also marked gpu; deselect with -m 'gpu and not perf')")


def _gpu_available():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture
def stream_beside():
    """``f(*streams)``: a stream whose work has been seen to run while a launch on each of ``streams`` waits.  The streams of a process share a few hardware
    queues, and two that share one run in order: whether a fresh stream shares another's depends on how many there were before it."""
    import torch
    from meshslice_amd import TensorParallel as TP

    def find(*streams):
        dev = streams[0].device
        torch.cuda.synchronize(dev)
        for _ in range(12):
            other = torch.cuda.Stream(dev)
            for cur in streams:
                with torch.cuda.stream(cur):
                    if not TP._runs_beside(cur, other, dev):
                        break
            else:
                torch.cuda.synchronize(dev)
                return other
        pytest.skip("no stream runs beside a waiting launch on this machine")
    return find


def pytest_collection_modifyitems(config, items):
    if _gpu_available():
        return
    skip = pytest.mark.skip(reason="no GPU in this process")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)
