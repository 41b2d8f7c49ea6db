"""Host: the Python shim of the engines tells torch's allocator about every gradient tensor it kept for a deferred cycle
before it lets go of it (the applying call has only been enqueued).  The library is stood in for."""
from types import SimpleNamespace

import pytest

import mxopt as mx


class Gradient:
    is_cuda = True

    def __init__(self):
        self.recorded = []

    def record_stream(self, stream):
        self.recorded.append(stream)


@pytest.mark.parametrize("call", ["flush_gradients", "reset"])
def test_gradients_of_a_deferred_cycle_are_recorded_before_they_are_dropped(call):
    eng = mx.SFTEngineOptimizerSide.__new__(mx.SFTEngineOptimizerSide)
    ok = lambda *a: 0
    eng.lib = SimpleNamespace(mxopt_engine_flush_gradients=ok, mxopt_engine_reset=ok, mxopt_engine_free=ok)
    eng.ctx, eng.handle, eng.defers = SimpleNamespace(handle=None, stream="the context's stream"), None, True
    held = [Gradient() for _ in range(3)]
    eng._held = [held[:2], held[2:]]
    getattr(eng, call)()
    assert [g.recorded for g in held] == [["the context's stream"]] * 3 and eng._held == []
