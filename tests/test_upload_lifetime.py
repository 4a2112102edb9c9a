"""Host arrays of queued uploads stay alive until the stream has been waited for (no GPU: the library is a stub)."""
import weakref

import numpy as np
import pytest

from trajectories import _native as N
from trajectories import configs
from trajectories.compile import compile_elements
from trajectories.device import Context
from trajectories.engine import Engine


class Stub:
    """Answers every entry point with success and notes which host arrays were alive at each wait."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return 0
        return call


@pytest.fixture
def stubbed(monkeypatch):
    lib = Stub()
    monkeypatch.setattr(N, "lib", lambda: lib)
    ctx = Context(0)
    ctx.handle = 1
    yield lib, ctx
    ctx.handle = None


def test_an_error_between_uploads(stubbed):
    lib, ctx = stubbed
    bl = configs.config0()
    eng = Engine(compile_elements(bl.elements, bl.g), ctx)
    first = np.arange(4.0)
    alive = weakref.ref(first)
    with pytest.raises(ValueError):
        eng.propagate(first, ["no number"] * 4, *np.zeros((4, 4)))
    del first
    assert "ctraj_memcpy" in lib.calls and "ctraj_sync" not in lib.calls  # its upload is queued
    assert alive() is not None
    ctx.sync()
    assert alive() is None


def test_a_failed_wait_keeps_them(stubbed, monkeypatch):
    lib, ctx = stubbed
    host = np.arange(4.0)
    alive = weakref.ref(host)
    ctx.scratch_from(host)
    del host
    with monkeypatch.context() as m:
        m.setattr(ctx, "handle", 2)
        lib.ctraj_sync = lambda handle: -2 if handle == 2 else 0
        lib.ctraj_last_error = lambda handle: b"stub"
        with pytest.raises(N.NativeError):
            ctx.sync()
    assert alive() is not None
    ctx.sync()
    assert alive() is None


def test_a_wait_inside_the_list(stubbed):
    """A collection may run anywhere, also where the list is changed, and its finalizers may wait for the stream."""
    lib, ctx = stubbed
    with ctx._uploads_lock:
        ctx.sync()
    assert "ctraj_sync" in lib.calls
