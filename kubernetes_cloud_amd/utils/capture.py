"""HIP-graph capture with Python's cyclic collector held off."""
from __future__ import annotations

import contextlib
import gc
import threading

import torch

_lock = threading.Lock()
_open = 0          # captures under way, in all threads
_enabled = False   # whether the collector was on before the first of them


@contextlib.contextmanager
def no_collection():
    """No automatic collection of reference cycles inside, on any thread (nests, and several threads may be inside).

    The collector runs in whichever thread's allocation crosses its threshold, so a capturing thread would run the
    destructors of whatever died in a cycle: a graph waits for the device when it goes, a pinned buffer records an event on
    the streams that used it. HIP refuses such calls to a thread that captures, and an error inside a destructor ends the
    process (SIGABRT) instead of raising."""
    global _open, _enabled
    with _lock:
        if _open == 0:
            _enabled = gc.isenabled()
            gc.disable()
        _open += 1
    try:
        yield
    finally:
        with _lock:
            _open -= 1
            if _open == 0 and _enabled:
                gc.enable()


@contextlib.contextmanager
def graph(g: torch.cuda.CUDAGraph, **kw):
    """``torch.cuda.graph`` without collections while it records, in thread-local mode: the RCCL process-group watchdog thread
    polls its work events while a capture runs; under the default global mode that query fails ("operation not permitted
    when stream is capturing") and the watchdog aborts the process."""
    with no_collection(), torch.cuda.graph(g, capture_error_mode="thread_local", **kw):
        yield


__all__ = ["graph", "no_collection"]
