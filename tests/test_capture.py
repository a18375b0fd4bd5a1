"""Graph captures run with the cyclic garbage collector off."""

import gc
import inspect
import threading
import weakref
from types import SimpleNamespace

import pytest
import torch

from kvengine_amd import engine, speculative
from kvengine_amd.capture import no_gc


def test_no_gc_turns_collection_off_and_back():
    assert gc.isenabled()
    with no_gc():
        assert not gc.isenabled()
        with no_gc():
            assert not gc.isenabled()
        assert not gc.isenabled()
    assert gc.isenabled()
    with pytest.raises(RuntimeError):
        with no_gc():
            raise RuntimeError("a capture that failed")
    assert gc.isenabled()


def test_no_gc_leaves_a_disabled_collector_disabled():
    gc.disable()
    try:
        with no_gc():
            assert not gc.isenabled()
        assert not gc.isenabled()
    finally:
        gc.enable()


def test_overlapping_captures_of_threads_end_with_collection_on():
    inside, leave = threading.Event(), threading.Event()

    def other():
        with no_gc():
            inside.set()
            leave.wait(10)

    t = threading.Thread(target=other)
    with no_gc():
        t.start()
        assert inside.wait(10)
    assert not gc.isenabled()  # the other thread still captures
    leave.set()
    t.join()
    assert gc.isenabled()


def test_every_capture_of_the_package_holds_collection_off():
    for module in (engine, speculative):
        lines = inspect.getsource(module).splitlines()
        captures = [s for s in lines if "torch.cuda.graph(" in s]
        assert captures and all("no_gc()" in s for s in captures), captures


def test_a_new_entry_of_iteration_graphs_collects_nothing(monkeypatch):
    """A first call on new models and pools, while another thread captures, must
    not run the collector: what it frees may hold graphs. (A full collection
    would also cost the call 60-90 ms.)"""
    class Obj(SimpleNamespace):
        __hash__ = object.__hash__

    def pool():
        return Obj(**{n: torch.zeros(1) for n in ("tables", "lens", "k", "v")})

    monkeypatch.setattr(speculative, "_GRAPHS", {})
    monkeypatch.setattr(speculative._IterationGraphs, "__init__", lambda self, pool, k: None)
    inside, leave = threading.Event(), threading.Event()

    def capture():
        with no_gc():
            inside.set()
            leave.wait(10)

    t = threading.Thread(target=capture)
    t.start()
    assert inside.wait(10)
    try:
        dead = Obj()
        dead.me = dead  # a cycle, as a dead pool's graphs can be in
        alive = weakref.ref(dead)
        del dead
        models = torch.nn.Linear(2, 2), torch.nn.Linear(2, 2)
        caches = Obj(pool=pool()), Obj(pool=pool())
        made = speculative._IterationGraphs.for_call(*models, *caches, 4)
        assert alive() is not None
        assert speculative._IterationGraphs.for_call(*models, *caches, 4) is made
    finally:
        leave.set()
        t.join()
    gc.collect()
    assert alive() is None
