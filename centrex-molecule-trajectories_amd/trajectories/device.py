"""Device context and buffers on top of libctraj.so.

Device memory is owned by :class:`DeviceArray` objects allocated through the library
(``ctraj_dev_alloc``); copies and kernels are queued on the context's single HIP stream.
"""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np

from . import _native as N


class DeviceArray:
    """A 1-D device buffer of ``n`` elements of ``dtype`` (owned; freed on ``free()``/GC)."""

    __slots__ = ("ctx", "n", "dtype", "nbytes", "ptr", "__weakref__")

    def __init__(self, ctx: "Context", n: int, dtype=np.float64):
        self.ctx = ctx
        self.n = int(n)
        self.dtype = np.dtype(dtype)
        self.nbytes = self.n * self.dtype.itemsize
        p = C.c_void_p()
        N.check("ctraj_dev_alloc", N.lib().ctraj_dev_alloc(ctx.handle, self.nbytes, C.byref(p)), ctx.handle)
        self.ptr = p.value

    def upload(self, host: np.ndarray, sync: bool = True):
        a = np.ascontiguousarray(host, dtype=self.dtype).reshape(-1)
        if a.size != self.n:
            raise ValueError(f"size mismatch {a.size} != {self.n}")
        self.ctx.memcpy(self.ptr, a.ctypes.data, self.nbytes, N.H2D)
        if sync:
            self.ctx.sync()
        return self

    def to_host(self, out: np.ndarray | None = None, count: int | None = None) -> np.ndarray:
        """Copy the buffer (or its first ``count`` elements) to the host."""
        k = self.n if count is None else max(0, min(int(count), self.n))
        if out is None:
            out = np.empty(k, dtype=self.dtype)
            self.ctx.read((self, out))
            return out
        if k:
            self.ctx.memcpy(out.ctypes.data, self.ptr, k * self.dtype.itemsize, N.D2H)
        self.ctx.sync()
        return out

    def fill(self, value):
        if self.dtype.itemsize == 8:
            bits = np.array([value], dtype=self.dtype).view(np.int64)[0]
            N.check("ctraj_fill_i64", N.lib().ctraj_fill_i64(self.ctx.handle, self.ptr, int(bits), self.n),
                    self.ctx.handle)
        elif self.dtype.itemsize == 1:
            N.check("ctraj_fill_u8", N.lib().ctraj_fill_u8(self.ctx.handle, self.ptr, int(value), self.nbytes),
                    self.ctx.handle)
        else:
            raise TypeError("fill supports 1- and 8-byte dtypes")
        return self

    def free(self):
        if self.ptr and self.ctx.handle:
            N.lib().ctraj_dev_free(self.ctx.handle, self.ptr)
        self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass

    def __len__(self):
        return self.n


class ScratchArray(DeviceArray):
    """A DeviceArray from the context's kept blocks, for buffers that live and die inside one call: they are used
    on the context's stream only and never handed to the caller (a freed block goes to the next request without
    waiting for the device; hipMalloc and hipFree took 3 ms of a 7 ms run_simulation)."""

    __slots__ = ()
    _pool = "scratch"

    def __init__(self, ctx: "Context", n: int, dtype=np.float64):
        self.ctx = ctx
        self.n = int(n)
        self.dtype = np.dtype(dtype)
        self.nbytes = self.n * self.dtype.itemsize
        p = C.c_void_p()
        name = f"ctraj_{self._pool}_alloc"
        N.check(name, getattr(N.lib(), name)(ctx.handle, self.nbytes, C.byref(p)), ctx.handle)
        self.ptr = p.value

    def free(self):
        if self.ptr and self.ctx.handle:
            getattr(N.lib(), f"ctraj_{self._pool}_free")(self.ctx.handle, self.ptr)
        self.ptr = None


class ResultArray(ScratchArray):
    """A DeviceArray for the caller, on any stream: given back, its block is kept, and handed out again only after the
    device has been waited for."""

    __slots__ = ()
    _pool = "result"


class Context:
    """One device + one HIP stream (``ctraj_ctx``)."""

    PINNED = 1 << 20  # bytes of page-locked memory that small results pass through

    def __init__(self, device: int = 0):
        L = N.lib()
        h = C.c_void_p()
        rc = L.ctraj_ctx_create(int(device), C.byref(h))
        if rc != N.OK:
            raise N.NativeError("ctraj_ctx_create", rc, L.ctraj_last_error(None).decode(errors="replace"))
        self.handle = h.value
        self.device = int(device)
        ncu, lds, wave, arch = (C.c_int32() for _ in range(4))
        N.check("ctraj_device_info",
                L.ctraj_device_info(self.handle, C.byref(ncu), C.byref(lds), C.byref(wave), C.byref(arch)),
                self.handle)
        self.n_cu, self.lds_per_block, self.wave, self.arch = ncu.value, lds.value, wave.value, arch.value
        self.bound = None  # the CompiledBeamline currently set on the device
        self.lock = threading.RLock()
        self._pinned = None  # (address, uint8 view), made on first use
        self._uploads, self._uploads_lock = [], threading.RLock()  # host arrays whose copies are queued

    # --- memory ---
    def alloc(self, n, dtype=np.float64) -> DeviceArray:
        return DeviceArray(self, n, dtype)

    def to_device(self, host, dtype=None) -> DeviceArray:
        host = np.asarray(host)
        d = DeviceArray(self, host.size, dtype or host.dtype)
        return d.upload(host)

    def scratch(self, n, dtype=np.float64) -> ScratchArray:
        return ScratchArray(self, n, dtype)

    def result(self, n, dtype=np.float64) -> ResultArray:
        return ResultArray(self, n, dtype)

    def trim(self) -> None:
        """Release the kept blocks of scratch and results (at most 1 and 8 GiB), for another allocator's use; the
        library's own allocations on this device do so by themselves where memory runs out."""
        N.check("ctraj_trim", N.lib().ctraj_trim(self.handle), self.handle)

    def scratch_from(self, host, dtype=None) -> ScratchArray:
        """Queue the upload of a host array into a scratch buffer.  The context holds the array until it has waited
        for the stream, whatever becomes of the caller (an error between this upload and the wait included)."""
        host = np.ascontiguousarray(host, dtype=dtype)
        d = ScratchArray(self, host.size, host.dtype)
        try:
            return d.upload(host, sync=False)
        finally:
            with self._uploads_lock:
                self._uploads.append(host)

    def read(self, *pairs) -> None:
        """Fill host arrays from device memory, pairs of (buffer or address, contiguous array), with one wait: small
        ones through page-locked memory, so that their copies are queued one after the other."""
        with self.lock:
            if self._pinned is None:
                p = C.c_void_p()
                N.check("ctraj_host_alloc", N.lib().ctraj_host_alloc(self.handle, self.PINNED, C.byref(p)), self.handle)
                self._pinned = (p.value, np.frombuffer((C.c_char * self.PINNED).from_address(p.value), np.uint8))
            base, view = self._pinned
            off, staged = 0, []
            try:
                for src, out in pairs:
                    src, nbytes = N.addr(src), out.nbytes
                    if not nbytes:
                        continue
                    if off + nbytes <= self.PINNED:
                        self.memcpy(base + off, src, nbytes, N.D2H)
                        staged.append((off, nbytes, out))
                        off += (nbytes + 63) & ~63
                    else:
                        self.memcpy(out.ctypes.data, src, nbytes, N.D2H)
            finally:  # no copy into the caller's arrays is left queued
                self.sync()
            for o, nbytes, out in staged:
                out.reshape(-1).view(np.uint8)[:] = view[o:o + nbytes]

    def memcpy(self, dst: int, src: int, nbytes: int, kind: int):
        N.check("ctraj_memcpy", N.lib().ctraj_memcpy(self.handle, dst, src, int(nbytes), int(kind)), self.handle)

    def sync(self):
        with self._uploads_lock:
            uploads, self._uploads = self._uploads, []
        try:
            N.check("ctraj_sync", N.lib().ctraj_sync(self.handle), self.handle)
        except BaseException:
            with self._uploads_lock:
                self._uploads += uploads
            raise

    # --- timing on the context stream ---
    def event_record(self, slot: int):
        N.check("ctraj_event_record", N.lib().ctraj_event_record(self.handle, int(slot)), self.handle)

    def event_elapsed_ms(self, a: int, b: int) -> float:
        ms = C.c_float()
        N.check("ctraj_event_elapsed", N.lib().ctraj_event_elapsed(self.handle, int(a), int(b), C.byref(ms)),
                self.handle)
        return float(ms.value)

    def phase_times(self, max_n: int = 64):
        """Kernel times (ms) of the launches made with RUN_PHASE_TIMES since the last call, oldest first:
        (walk to the lens, lens, walk after the lens) arrays; a single-kernel run has all its time in the
        lens array."""
        bufs = [(C.c_float * max_n)() for _ in range(3)]
        cnt = C.c_int32()
        N.check("ctraj_phase_times", N.lib().ctraj_phase_times(self.handle, int(max_n), *bufs, C.byref(cnt)),
                self.handle)
        k = cnt.value
        return tuple(np.array(b[:k], dtype=np.float64) for b in bufs)

    def close(self):
        if getattr(self, "handle", None):
            if self._pinned is not None:
                N.lib().ctraj_host_free(self.handle, self._pinned[0])
                self._pinned = None
            N.lib().ctraj_ctx_destroy(self.handle)
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


_DEFAULT: dict[int, Context] = {}
_LOCK = threading.Lock()


def get_context(device: int = 0) -> Context:
    """Process-wide context for ``device`` (created on first use)."""
    with _LOCK:
        ctx = _DEFAULT.get(device)
        if ctx is None or ctx.handle is None:
            ctx = Context(device)
            _DEFAULT[device] = ctx
        return ctx
