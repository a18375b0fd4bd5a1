"""Garbage collection held off while a HIP graph is being captured.

Destroying a captured graph synchronizes the device, which is an error while
another capture is under way, and in a destructor that error ends the process.
Python's cyclic collector runs whenever enough objects have been allocated, so
a dead engine, pool or model that holds graphs in a reference cycle could be
collected in the middle of a capture.
"""

from __future__ import annotations

import contextlib
import gc
import threading

_LOCK = threading.Lock()
_depth = 0          # captures under way, over all threads
_was_enabled = False


@contextlib.contextmanager
def no_gc():
    """Automatic garbage collection is off inside, and back as it was once the
    last of the overlapping users has left."""
    global _depth, _was_enabled
    with _LOCK:
        if _depth == 0:
            _was_enabled = gc.isenabled()
            gc.disable()
        _depth += 1
    try:
        yield
    finally:
        with _LOCK:
            _depth -= 1
            if _depth == 0 and _was_enabled:
                gc.enable()
