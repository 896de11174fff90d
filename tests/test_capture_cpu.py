"""No reference cycle is collected while a HIP graph is being captured: a stand-in for the capture on the CPU, a dead cycle with
a finalizer, and allocations past every threshold of the collector."""
import contextlib
import gc
import threading
from types import SimpleNamespace

import pytest
import torch

from kubernetes_cloud_amd.utils import capture


class _Dead:
    """An object in a cycle of its own; notes whether it went during a capture."""
    recording = False
    went = []

    def __init__(self):
        self.me = self

    def __del__(self):
        _Dead.went.append(_Dead.recording)


def _work(*_, **__):
    """What a captured step does on the host, and more: a dead cycle, then allocations past the thresholds."""
    for _ in range(3):
        _Dead()
        keep = [[] for _ in range(200_000)]
    return keep[0]


@pytest.fixture
def fakes(monkeypatch):
    @contextlib.contextmanager
    def record(g, pool=None, stream=None, capture_error_mode="global"):
        assert capture_error_mode == "thread_local"
        _Dead.recording = True
        yield
        _Dead.recording = False

    stream = SimpleNamespace(wait_stream=lambda s: None)
    for name, value in dict(graph=record, CUDAGraph=object, Stream=lambda *a, **k: stream, current_stream=lambda *a: stream,
                            stream=lambda s: contextlib.nullcontext(), graph_pool_handle=lambda: (0, 0)).items():
        monkeypatch.setattr(torch.cuda, name, value)
    gc.collect()
    _Dead.went, _Dead.recording = [], False
    yield
    gc.collect()
    assert _Dead.went and not any(_Dead.went)  # all of them went, none during a capture
    assert gc.isenabled()


def test_step_capture(fakes):
    from kubernetes_cloud_amd.engine.runner import StepRunner
    r = SimpleNamespace(_step_state=lambda: [], _capture_stream=None, _pool=None, _graphs={}, _step_body=_work)
    StepRunner._capture(r, {}, 1, 256)
    assert list(r._graphs) == [(1, 256, False)]


def test_unet_capture(fakes):
    from kubernetes_cloud_amd.models.sd_pipeline import UNetGraph
    x = torch.zeros(1)
    assert UNetGraph(lambda *a: _work())._capture(x, x, x) is not False


def test_nested_failing_and_concurrent_captures(fakes):
    inside, leave = threading.Event(), threading.Event()

    def other():
        with capture.no_collection():
            inside.set()
            leave.wait(10)

    t = threading.Thread(target=other)
    t.start()
    assert inside.wait(10)
    with pytest.raises(KeyError):
        with capture.no_collection():
            with capture.no_collection():
                _work()
            raise KeyError
    assert not gc.isenabled()  # the other thread still captures
    leave.set()
    t.join()
    assert gc.isenabled()


def test_a_collector_that_is_off_stays_off():
    gc.disable()
    try:
        with capture.no_collection():
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()


@pytest.mark.parametrize("family", ["megusun", "rezusun", "begopel", "gibipel"])
def test_runners_go_with_their_last_reference(family):
    """No cycle holds a runner's cache, graphs and pinned buffers until a collection."""
    import importlib
    import weakref

    from kubernetes_cloud_amd.engine.llm_engine import LLMEngine, SamplingParams
    t = importlib.import_module("tests.test_" + family)
    for name in t.CFGS:
        m = t.make(t.CFGS[name] if family == "megusun" else name, "cpu", torch.float32)[0]
        gc.collect()
        gc.disable()
        try:
            e = LLMEngine(m, max_slots=2, max_len=64)
            e.generate([[1, 2, 3]], SamplingParams(max_new_tokens=3, do_sample=False))
            left = weakref.ref(e.runner)
            del e
            assert left() is None, name
        finally:
            gc.enable()
