"""Graph captures run with the cyclic garbage collector off."""

import gc
import inspect
import threading

import pytest

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
