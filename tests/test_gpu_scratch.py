"""GPU: scratch blocks are exclusive while held, reused after they are given back, and bounded."""
import ctypes as C
import threading

import numpy as np
import pytest

from trajectories import _native as N
from trajectories import configs
from trajectories.device import Context
from trajectories.engine import Engine
from trajectories.stream import StreamedRun

pytestmark = pytest.mark.gpu


def test_blocks():
    ctx = Context(0)
    a = ctx.scratch(1000)
    p = a.ptr
    b = ctx.scratch(1000)
    assert b.ptr != p
    a.free()
    assert ctx.scratch(990).ptr == p  # the block given back
    with pytest.raises(N.NativeError):
        N.check("ctraj_scratch_free", N.lib().ctraj_scratch_free(ctx.handle, b.ptr + 8), ctx.handle)
    big = ctx.scratch((3 << 30) // 8)  # larger than everything that is kept: released at once
    big.free()
    h = np.arange(300_000.0)  # through page-locked memory and past it
    d, e = ctx.scratch_from(h), ctx.scratch_from(h[:5])
    ctx.sync()
    x, y, z = np.empty_like(h), np.empty(5), np.empty(0)
    ctx.read((d, x), (e, y), (d, z))
    assert np.array_equal(x, h) and np.array_equal(y, h[:5])
    ctx.close()


def test_threads_hold_different_blocks():
    ctx = Context(0)
    seen, lock, bad = set(), threading.Lock(), []

    def work():
        for n in (10, 1000, 5000) * 30:
            a = ctx.scratch(n)
            with lock:
                if a.ptr in seen:
                    bad.append(a.ptr)
                seen.add(a.ptr)
            with lock:
                seen.discard(a.ptr)
            a.free()

    ts = [threading.Thread(target=work) for _ in range(6)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
    ctx.close()


def test_results_do_not_depend_on_reused_blocks():
    eng = Engine(configs.config1())
    X, V = configs.draw_source(30_000, 3)
    first = {n: eng.propagate(*X[:, :n], *V[:, :n], aoi_labels=["Detected"]) for n in (30_000, 1, 777)}
    for n in (777, 30_000, 1):
        r = eng.propagate(*X[:, :n], *V[:, :n], aoi_labels=["Detected"])
        assert np.array_equal(r["label"], first[n]["label"]) and np.array_equal(r["tally"], first[n]["tally"])
        assert all(np.array_equal(r["out"][k], first[n]["out"][k]) for k in r["out"])
        assert np.array_equal(np.sort(r["aoi_index"]), np.sort(first[n]["aoi_index"]))


@pytest.mark.parametrize("old", [1, 3, 4])
def test_a_full_pool_keeps_the_blocks_in_use(old):
    """Blocks of sizes no longer asked for make room: a block given back last is there for the next request,
    however many older ones the pool (1 GiB) holds."""
    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert N.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # of the runtime the library uses
        return free.value

    ctx = Context(0)
    mib = (1 << 20) // 8
    for b in [ctx.scratch(n * mib) for n in (240, 200, 220, 260)[:old]]:
        b.free()
    for _ in range(3):
        big = ctx.scratch(640 * mib)
        big.free()
        free = free_bytes()
        big = ctx.scratch(640 * mib)
        assert free - free_bytes() < 64 << 20  # it was kept
        big.free()
    held = free_bytes()
    ctx.close()
    assert free_bytes() - held < (1 << 30) + (64 << 20)  # what the pool held is bounded


def test_results_outlive_their_run_and_are_kept():
    """A result held by the caller is not handed out again, its dropped block is (also after use on another
    stream: giving it back waits for the device), and blocks beyond what is kept are released."""
    run = StreamedRun(configs.config4(), 60_000, chunk=1 << 20, seed=3, n_states=4)
    a = run.run()
    want = a.trajectories.to_host()
    b = run.run()
    assert b.trajectories.ptr != a.trajectories.ptr
    assert np.array_equal(a.trajectories.to_host(), want, equal_nan=True)
    p, ctx = a.trajectories.ptr, a.trajectories.ctx
    del a
    c = run.run()
    assert c.trajectories.ptr == p
    assert np.array_equal(c.trajectories.to_host(), want, equal_nan=True)
    with pytest.raises(N.NativeError):  # of the other kind
        N.check("ctraj_scratch_free", N.lib().ctraj_scratch_free(ctx.handle, p), ctx.handle)
    big = ctx.result((9 << 30) // 8)
    big.free()
    ctx.result((9 << 30) // 8).free()
