"""Captured graphs are not destroyed while another is captured: their destructor waits for the device, which a capture does not allow.
Torch's graphs stand-ins here, which say when they go."""
import contextlib
import ctypes
import gc
import threading

import pytest
import torch

_kept = []  # destructors: a failed test's frames may outlive it


@pytest.fixture
def cuda(monkeypatch):
    """Captures without a GPU. ``gone``: for every graph that was destroyed, whether some capture was under way; ``inside``: called in every
    capture."""
    class Fake:
        gone, inside, here = [], staticmethod(lambda: None), 0

    # what goes with its last reference, like a C++ object, and not when the collector finds it: a capsule's destructor
    destroyed = ctypes.CFUNCTYPE(None, ctypes.c_void_p)(lambda _: Fake.gone.append(Fake.here > 0))
    _kept.append(destroyed)
    capsule = ctypes.PYFUNCTYPE(ctypes.py_object, ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p)(("PyCapsule_New", ctypes.pythonapi))

    class Graph:
        def __init__(self):
            self.native, self.replays = capsule(1, None, ctypes.cast(destroyed, ctypes.c_void_p)), 0

        def replay(self):
            self.replays += 1

    @contextlib.contextmanager
    def graph(g, pool=None):
        Fake.here += 1
        try:
            Fake.inside()
            yield
        finally:
            Fake.here -= 1

    class Stream:
        def __init__(self, *a, **k):
            pass

        def wait_stream(self, other):
            pass

    empty = torch.empty
    for name, f in (("CUDAGraph", Graph), ("graph", graph), ("is_current_stream_capturing", lambda: Fake.here > 0), ("Stream", Stream),
                    ("stream", lambda s: contextlib.nullcontext()), ("current_stream", Stream), ("synchronize", lambda *a: None),
                    ("graph_pool_handle", lambda: None)):
        monkeypatch.setattr(torch.cuda, name, f)
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: empty(*a, **k))
    gc.collect()
    yield Fake
    gc.collect()


def _captured(name):
    from llmd_amd.engine.config import EngineConfig
    from llmd_amd.engine.engine import LLMEngine

    cfg = EngineConfig.create(name, device="cpu", dtype="bfloat16", block_size=64, num_gpu_blocks=8, max_num_seqs=2, max_model_len=200,
                              max_num_batched_tokens=64, enable_prefix_caching=False)
    runner = LLMEngine(cfg).runner
    runner.is_gpu = True
    runner.capture_graphs()
    return runner


@pytest.mark.parametrize("name", ["tiny-kokatar", "tiny-llama"])  # per-layer stacks, the other models
def test_a_runner_in_a_cycle(cuda, name):
    first = _captured(name)
    n = len(first.graphs)
    first.me = first
    del first
    assert n >= 2 and not cuda.gone
    cuda.inside = gc.collect  # as the collector may come at any allocation
    second = _captured(name)
    cuda.inside = lambda: None
    assert cuda.gone == [False] * n  # all of them, and none during a capture
    next(iter(second.graphs.values()))[0].replay()
    second.graphs.clear()
    assert cuda.gone == [False] * 2 * n


def test_somebody_elses_capture(cuda):
    from llmd_amd.engine.step_graph import StepGraph

    g, other = StepGraph(), StepGraph()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        del g
        assert cuda.gone == []
    other.replay()  # what was left goes with the next use
    assert cuda.gone.count(False) >= 1 and True not in cuda.gone and other.graph.replays == 1


def test_a_capture_in_another_thread(cuda):
    from llmd_amd.engine.step_graph import StepGraph

    g, inside, done = StepGraph(), threading.Event(), threading.Event()

    def capture():
        with StepGraph().capture():
            inside.set()
            done.wait(10)

    t = threading.Thread(target=capture)
    t.start()
    inside.wait(10)
    del g
    n = len(cuda.gone)
    done.set()
    t.join()
    assert n == 0 and cuda.gone == [False, False]


def test_a_failed_capture(cuda):
    from llmd_amd.engine.step_graph import StepGraph

    with pytest.raises(ValueError):
        with StepGraph().capture():
            raise ValueError
    g = StepGraph()
    del g
    assert True not in cuda.gone and len(cuda.gone) == 2
