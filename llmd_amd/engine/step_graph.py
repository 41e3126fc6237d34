"""A step's captured graph, destroyed only where no capture is under way.

On ROCm a graph's destructor waits for the device, which is refused while a stream is being captured, and an error in a destructor
ends the process (SIGABRT, without a fault of the GPU). A runner whose last references form a cycle - somebody's closure over one of its
methods in its own attributes is enough - is destroyed by the cyclic collector, which may run at any allocation, also among those of
the model's Python code while the next runner captures; ``torch.cuda.graph`` does not collect before it begins.
"""
from __future__ import annotations

import contextlib
import sys
import threading

import torch


class _Leaving:
    """Graphs whose owners are gone. They are destroyed under the lock under which captures begin."""

    def __init__(self):
        self.lock, self.captures, self.graphs = threading.Lock(), 0, []

    def release(self):
        # (never waits: the collector may have interrupted the lock's holder. What is left goes with a later call.)
        if self.lock.acquire(blocking=False):
            try:
                if not self.captures and not torch.cuda.is_current_stream_capturing():
                    self.graphs.clear()
            finally:
                self.lock.release()

    def count(self, by: int):
        with self.lock:
            self.captures += by


_leaving = _Leaving()


class StepGraph:
    def __init__(self):
        self.graph = torch.cuda.CUDAGraph()

    @contextlib.contextmanager
    def capture(self, pool=None):
        _leaving.release()
        _leaving.count(1)
        try:
            with torch.cuda.graph(self.graph, pool=pool):
                yield
        finally:
            _leaving.count(-1)
            _leaving.release()

    def replay(self):
        if _leaving.graphs:
            _leaving.release()
        self.graph.replay()

    def __del__(self, leaving=_leaving, finalizing=sys.is_finalizing):
        graph = self.__dict__.pop("graph", None)
        if graph is not None and not finalizing():
            leaving.graphs.append(graph)
            del graph
            leaving.release()
