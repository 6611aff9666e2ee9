"""Graph capture with the garbage collector held off."""
from __future__ import annotations

import contextlib
import gc
import threading

import torch

_lock = threading.Lock()
_captures = 0
_was_enabled = False


@contextlib.contextmanager
def capture_graph(graph: "torch.cuda.CUDAGraph", **kw):
    """``torch.cuda.graph`` without collections inside it.  A collection that happens to start during the capture may
    free an engine dropped earlier (engines and their buffers refer to each other), and with it a CUDAGraph, whose
    destructor on ROCm waits for the device -- not permitted while a stream captures, and an error in a destructor ends
    the process.  (torch itself collected before every capture once; 2.10 does not.)  Captures on several threads share
    the hold: the collector runs again after the last one."""
    global _captures, _was_enabled
    with _lock:
        if _captures == 0:
            _was_enabled = gc.isenabled()
            gc.disable()
        _captures += 1
    try:
        with torch.cuda.graph(graph, **kw):
            yield
    finally:
        with _lock:
            _captures -= 1
            if _captures == 0 and _was_enabled:
                gc.enable()
