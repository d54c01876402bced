"""When captured decode graphs are freed (CPU; stubs stand in for the GPU).

A graph's destructor waits for the device, which is refused while a stream is
capturing, and the process ends: graphs of an engine that is gone must never be
freed inside a capture."""

from __future__ import annotations

import contextlib
import gc
import sys
import threading
import weakref
from types import SimpleNamespace

import pytest
import torch

from litevllm import workloads
from litevllm.config.config import (CacheConfig, EngineConfig, ModelConfig, SchedulerConfig)
from litevllm.engine import model_runner as mr


class Gpu:
    """torch.cuda's capture calls; `capturing` holds the threads inside one.
    Live graphs are counted by the references they hold to one plain object:
    like a C++ member it goes when a graph is freed, not when it is garbage."""

    def __init__(self, monkeypatch, forward):
        self.capturing, self.freed_in_capture = set(), 0
        self.forward, self.member = forward, object()
        stream = SimpleNamespace(wait_stream=lambda s: None)
        gpu = self
        self.none_alive = 0
        self.none_alive = self.alive()

        class Graph:
            def __init__(self):
                self.member = gpu.member

        @contextlib.contextmanager
        def graph(g, pool=None):
            before = gpu.alive()
            gpu.capturing.add(threading.get_ident())
            try:
                yield
            finally:
                gpu.capturing.discard(threading.get_ident())
                gpu.freed_in_capture += before - gpu.alive()
        for name, fn in dict(
                graph_pool_handle=lambda: (0, 1), Stream=lambda: stream, graph=graph,
                current_stream=lambda *a: stream, stream=lambda s: contextlib.nullcontext(),
                CUDAGraph=Graph, synchronize=lambda: None,
                is_current_stream_capturing=lambda: threading.get_ident() in gpu.capturing,
        ).items():
            monkeypatch.setattr(torch.cuda, name, fn)
        monkeypatch.setattr(mr.ops, "pack_inputs", lambda *a, **k: None)

    def alive(self):
        return sys.getrefcount(self.member) - self.none_alive

    def runner(self):
        mc = ModelConfig(model="shape-only", dtype="bfloat16", max_model_len=64,
                         load_format="dummy", hf_overrides=dict(workloads.QWEN3_06B_SHAPE))
        mc.resolve()
        config = EngineConfig(model_config=mc, cache_config=CacheConfig(block_size=16),
                              scheduler_config=SchedulerConfig(max_num_seqs=4), device="cpu",
                              skip_tokenizer_init=True)
        r = mr.ModelRunner(config)
        r.model = lambda **k: self.forward()
        r.kv_cache = SimpleNamespace(num_layers=1, get_kv=lambda i: None)
        return r


@pytest.fixture
def plain_gc():
    """The collector on, with a heap small enough for full collections (they
    wait for a quarter of the older objects to be new)."""
    was, threshold = gc.isenabled(), gc.get_threshold()
    gc.freeze()
    gc.collect()
    yield
    gc.unfreeze()
    gc.set_threshold(*threshold)
    gc.enable() if was else gc.disable()


def _allocate():
    return [[i] for i in range(2000)] and torch.zeros(1)


def test_graphs_go_with_the_last_reference_to_their_runner(monkeypatch, plain_gc):
    gpu = Gpu(monkeypatch, _allocate)
    r = gpu.runner()
    r.capture_decode_graphs()
    assert gpu.alive() == len(r.graphs.graphs) >= 3
    gc.disable()
    gone = weakref.ref(r.graphs)
    del r
    assert gone() is None and gpu.alive() == 0


def test_no_collection_inside_a_capture(monkeypatch, plain_gc):
    """An engine that only the collector can free (a hook on its runner refers
    back to it) and that goes during a capture is freed after it."""
    gpu = Gpu(monkeypatch, _allocate)
    box = [gpu.runner()]
    box[0].capture_decode_graphs()
    n = gpu.alive()
    box[0].execute_model = lambda meta, r=box[0]: r

    def forward():
        if gpu.capturing:
            box.clear()
            gc.set_threshold(1, 1, 1)
        return _allocate()
    gpu.forward = forward
    new = gpu.runner()
    new.capture_decode_graphs()
    gc.collect()
    assert gc.isenabled() and gpu.freed_in_capture == 0 and gpu.alive() == n


def test_garbage_goes_before_a_capture(monkeypatch, plain_gc):
    gpu = Gpu(monkeypatch, _allocate)
    old = gpu.runner()
    old.capture_decode_graphs()
    n = gpu.alive()
    old.execute_model = lambda meta, r=old: r
    gc.disable()
    del old
    seen = []

    def forward():
        seen.append(gpu.alive())
        return _allocate()
    gpu.forward = forward
    new = gpu.runner()
    new.capture_decode_graphs()
    assert seen[0] == 0 and gpu.alive() == n and not gc.isenabled()


def test_graphs_dropped_inside_another_capture_are_kept_until_after(monkeypatch, plain_gc):
    """The collector may run in a capture the program makes itself."""
    gpu = Gpu(monkeypatch, _allocate)
    r = gpu.runner()
    r.capture_decode_graphs()
    n = gpu.alive()
    r.execute_model = lambda meta, r=r: r
    del r
    with torch.cuda.graph(None):
        gc.collect()
        assert gpu.alive() == n
    assert gpu.freed_in_capture == 0
    other = gpu.runner()
    other.capture_decode_graphs()
    assert gpu.alive() == n and not mr._retired
    other.release_decode_graphs()
    assert gpu.alive() == 0


def test_a_drop_on_another_thread_waits_for_the_capture(monkeypatch, plain_gc):
    started, box = threading.Event(), []

    def drop():
        started.wait(10)
        box.clear()
    thread = threading.Thread(target=drop)

    def forward():
        started.set()
        if gpu.capturing:
            thread.join(0.2)
        return torch.zeros(1)
    gpu = Gpu(monkeypatch, _allocate)
    box.append(gpu.runner())
    box[0].capture_decode_graphs()
    n = gpu.alive()
    new = gpu.runner()
    gpu.forward = forward
    thread.start()
    new.capture_decode_graphs()
    thread.join(10)
    assert not thread.is_alive() and gpu.freed_in_capture == 0 and gpu.alive() == n


def test_a_capture_that_fails_leaves_the_collector_on(monkeypatch, plain_gc):
    gpu = Gpu(monkeypatch, lambda: 1 // 0)
    with pytest.raises(ZeroDivisionError):
        gpu.runner().capture_decode_graphs()
    assert gc.isenabled()


def test_warm_up_and_capture_take_one_route(monkeypatch, plain_gc):
    """A library first used by a thread inside a capture makes its handle
    there, which the runtime does not survive: the forward that is captured and
    the one that warms up for it leave the same products to the library, on the
    capturing thread only."""
    native, seen = mr.ops._native(), []

    def state():
        was = native.library_products(True)
        native.library_products(was)
        return was

    def forward():
        other = []
        t = threading.Thread(target=lambda: other.append(state()))
        t.start()
        t.join(10)
        seen.append((bool(gpu.capturing), state(), other[0]))
        return torch.zeros(1)
    gpu = Gpu(monkeypatch, forward)
    gpu.runner().capture_decode_graphs()
    assert {c for c, _, _ in seen} == {False, True}
    assert all(on and not elsewhere for _, on, elsewhere in seen) and not state()
    gpu.forward = lambda: 1 // 0
    with pytest.raises(ZeroDivisionError):
        gpu.runner().capture_decode_graphs()
    assert not state()
