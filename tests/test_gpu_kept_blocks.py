"""GPU: what the kept blocks of a context take from the device's memory, and when they give it back."""
import ctypes as C

import pytest

from trajectories import _native as N
from trajectories.device import Context

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert N.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # of the runtime the library uses
    return free.value


@pytest.fixture
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("kind,nbytes", [("scratch", 3 * GIB // 2 + 80 * (1 << 20)), ("result", 35 * GIB // 2)])
def test_a_block_that_is_not_kept_takes_what_it_asks_for(ctx, kind, nbytes):
    before = free_bytes()
    b = getattr(ctx, kind)(nbytes // 8)
    assert before - free_bytes() <= nbytes + (4 << 20)  # the driver's own granularity
    b.free()
    assert free_bytes() >= before - (4 << 20)


@pytest.mark.parametrize("nbytes", [1 << 50, 1 << 63, (1 << 64) - 8])
def test_a_size_out_of_range_is_refused(ctx, nbytes):
    p = C.c_void_p()
    for kind in ("scratch", "result"):
        assert getattr(N.lib(), f"ctraj_{kind}_alloc")(ctx.handle, nbytes, C.byref(p)) == N.ENOMEM
        assert not p.value
        with pytest.raises(N.NativeError):
            getattr(ctx, kind)(-1)


@pytest.mark.parametrize("kind", ["scratch", "result"])
def test_kept_memory_is_there_for_others(ctx, kind):
    """A call releases what a context keeps, and so does an allocation of another context that finds no room."""
    nbytes, margin = 7 * GIB // 8, 8 << 20  # what else of the process comes and goes meanwhile
    other = Context(0)
    before = free_bytes()
    for release in (ctx.trim, lambda: pytest.raises(N.NativeError, other.alloc, 1 << 47)):
        getattr(ctx, kind)(nbytes // 8).free()
        assert free_bytes() <= before - nbytes + margin  # kept
        release()
        assert free_bytes() >= before - margin
    other.close()


def test_a_result_given_back_while_a_stream_is_captured(ctx):
    """As a garbage collection may: the capture goes on, and the block is there for the next request."""
    hip = N.lib()  # the runtime's own entry points, of the runtime the library uses
    stream, graph = C.c_void_p(), C.c_void_p()
    n = (64 << 20) // 8
    a = ctx.result(n)
    p = a.ptr
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    assert hip.hipStreamBeginCapture(stream, 0) == 0  # of any thread's calls
    a.free()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    assert ctx.result(n).ptr == p
