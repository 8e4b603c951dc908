"""HIP runtime and rocBLAS through ctypes: device memory, copies and FP64
products for the NumPy array family, which therefore needs no PyTorch.

The HIP runtime is reached by its soname after libozaki_amd.so has been
loaded, so this module and the library always share the one copy of the
runtime in the process (PyTorch ships one under the same soname; whichever
was loaded first serves both).  All work runs on the null stream, in order
with the library's kernels, which this family launches there too.

Device memory comes from a caching pool: blocks are rounded to size classes
and kept for reuse after their arrays are garbage collected, so repeated
calls of one shape allocate nothing after the first.

Host copies of 1 MiB and more go through pinned memory: the
library's host threads move bytes between the NumPy array and it while
others are on the link (a direct copy from pageable memory,
and the page faults of a fresh output array, are otherwise serial).
"""

import atexit
import ctypes
import os
import threading

import numpy as np

from . import _lib

_ROCM_LIB = "/opt/rocm/lib"
_H2D, _D2H, _D2D = 1, 2, 3
_COPY_UP, _COPY_DOWN, _COPY_UP_NEXT = 0, 1, 2  # ozk_copy_slots
_OP_N, _OP_T = 111, 112  # rocblas_operation_none / _transpose


def _open(soname):
    """The library of this soname already in the process, else ROCm's."""
    try:
        return ctypes.CDLL(soname)
    except OSError:
        return ctypes.CDLL(os.path.join(_ROCM_LIB, soname))


class _Runtime:
    def __init__(self):
        _lib.load()  # pulls libamdhip64.so.7 in through its runpath
        h = _open("libamdhip64.so.7")
        vp, sz, i = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int
        for name, args in [("hipMalloc", [ctypes.POINTER(vp), sz]), ("hipFree", [vp]),
                           ("hipMemcpy", [vp, vp, sz, i]),
                           ("hipMemset", [vp, i, sz]),
                           ("hipHostFree", [vp]),
                           ("hipStreamDestroy", [vp]),
                           ("hipDeviceSynchronize", []),
                           ("hipHostMalloc", [ctypes.POINTER(vp), sz, ctypes.c_uint]),
                           ("hipEventCreate", [ctypes.POINTER(vp)]),
                           ("hipEventRecord", [vp, vp]),
                           ("hipEventSynchronize", [vp]),
                           ("hipEventDestroy", [vp]),
                           ("hipStreamSynchronize", [vp]),
                           ("hipStreamCreateWithFlags", [ctypes.POINTER(vp), ctypes.c_uint]),
                           ("hipGetDeviceCount", [ctypes.POINTER(i)]),
                           ("hipGetDevice", [ctypes.POINTER(i)]),
                           ("hipGetLastError", [])]:
            fn = getattr(h, name)
            fn.restype = i
            fn.argtypes = args
        h.hipGetErrorString.restype = ctypes.c_char_p
        h.hipGetErrorString.argtypes = [i]
        self.h = h

    def check(self, rc, what):
        if rc != 0:
            msg = self.h.hipGetErrorString(rc).decode(errors="replace")
            self.h.hipGetLastError()  # leave no error behind for other users of the runtime
            raise _lib.OzakiError(f"{what} failed: {msg} ({rc})")

    def device_count(self):
        n = ctypes.c_int(0)
        rc = self.h.hipGetDeviceCount(ctypes.byref(n))
        if rc != 0:
            self.h.hipGetLastError()  # clear the sticky "no device" status
            return 0
        return n.value

    def device(self):
        d = ctypes.c_int(0)
        self.check(self.h.hipGetDevice(ctypes.byref(d)), "hipGetDevice")
        return d.value

    def malloc(self, nbytes):
        p = ctypes.c_void_p()
        self.check(self.h.hipMalloc(ctypes.byref(p), nbytes), f"hipMalloc({nbytes})")
        return p.value

    def free(self, ptr):
        self.check(self.h.hipFree(ptr), "hipFree")

    def copy(self, dst, src, nbytes, kind):
        if nbytes:
            self.check(self.h.hipMemcpy(dst, src, nbytes, kind), "hipMemcpy")

    def memset(self, dst, value, nbytes):
        if nbytes:
            self.check(self.h.hipMemset(dst, value, nbytes), "hipMemset")

    def sync(self, stream=None):
        self.check(self.h.hipStreamSynchronize(stream), "hipStreamSynchronize")

    def host_malloc(self, nbytes):
        p = ctypes.c_void_p()
        self.check(self.h.hipHostMalloc(ctypes.byref(p), nbytes, 0), f"hipHostMalloc({nbytes})")
        return p.value

    def host_free(self, p):
        self.check(self.h.hipHostFree(p), "hipHostFree")

    def event(self):
        e = ctypes.c_void_p()
        self.check(self.h.hipEventCreate(ctypes.byref(e)), "hipEventCreate")
        return e.value

    def record(self, e, stream=None):
        self.check(self.h.hipEventRecord(e, stream), "hipEventRecord")

    def nonblocking_stream(self):
        """A stream that does not wait for the null stream's work, nor the
        null stream for its (hipStreamNonBlocking), at the default priority."""
        s = ctypes.c_void_p()
        self.check(self.h.hipStreamCreateWithFlags(ctypes.byref(s), 1),
                   "hipStreamCreateWithFlags")
        return s.value

    def wait(self, e):
        self.check(self.h.hipEventSynchronize(e), "hipEventSynchronize")

    def destroy_event(self, e):
        self.check(self.h.hipEventDestroy(e), "hipEventDestroy")


# Host copies of at least _COPY_MIN bytes go through pinned memory
# (_Stager); smaller ones are as fast as the runtime's own copies.  So is an
# upload below _ALONE_MIN that no other follows or precedes, since staging gains
# from the overlap of two (host products of an array of 1, 2, 4, 8, 12 MiB with a
# small one: 177, 211, 321, 535, 715 us; staged 190, 240, 346, 490, 610).  Those
# above _SLOTS * _SLOT bytes take the larger slots.  Products whose halves reach
# _STAGE_MIN bytes run in two halves (matmul).
_COPY_MIN = 1 << 20
_ALONE_MIN = 6 << 20
ALONE, FIRST, FOLLOWING = 0, 1, 2  # place of an upload among several (from_numpy)
_SLOTS, _SLOT = 8, 4 << 20
_BIG_SLOTS, _BIG_SLOT = 4, 32 << 20
_STAGE_MIN = 32 << 20
_STAGE_CHUNK = 64 << 20


class _Slots:
    """Pinned slots with an event each (ozk_copy_slots).  The lock hands out
    the slot a transfer starts at."""

    def __init__(self, rt, slot, slots):
        self.slot, self.slots, self.first = int(slot), int(slots), 0
        self.buf = rt.host_malloc(self.slot * self.slots)
        self.ev = (ctypes.c_void_p * self.slots)(*[rt.event() for _ in range(self.slots)])
        self.lock = threading.Lock()

    def copy(self, way, dev_ptr, host, threads, stream):
        with self.lock:
            first = self.first
            self.first = (first + -(-host.nbytes // self.slot)) % self.slots
        _lib.check(_lib.load().ozk_copy_slots(
            way, dev_ptr, host.ctypes.data, host.nbytes, self.buf, self.slot, self.slots,
            first, self.ev, threads, stream))

    def release(self, h):
        h.hipHostFree(self.buf)
        for e in self.ev:
            h.hipEventDestroy(e)


class _Stager:
    """Pinned memory of the library's staged copies, allocated once per device
    and kept for the process: slots for the way up, as much memory with a
    flag word and a device counter per 512 KiB for the way down
    (ozk_copy_to_host), and larger slots for large transfers either way.  The
    library sees to it that transfers of several threads do not meet."""

    def __init__(self, rt, slot=_SLOT, slots=_SLOTS):
        self.rt, self.size = rt, int(slot) * int(slots)
        self.up, self.big = _Slots(rt, slot, slots), None
        self.down = rt.host_malloc(self.size)
        words = 4 * (self.size >> 19)
        self.flags, self.counts = rt.host_malloc(words), rt.malloc(words)
        rt.memset(self.counts, 0, words)
        rt.sync()
        ctypes.memset(self.flags, 0, words)
        for p in (self.up.buf, self.down):  # map the pages now, not call by call
            ctypes.memset(p, 0, self.size)
        self.max_threads = max(1, min(8, os.cpu_count() or 1))
        self.lock = threading.Lock()

    def _threads(self, nbytes):
        return min(self.max_threads, 1 + (nbytes >> 20))

    def _big(self):
        with self.lock:
            if self.big is None:
                self.big = _Slots(self.rt, _BIG_SLOT, _BIG_SLOTS)
            return self.big

    def to_device(self, dev_ptr, host, stream=None, following=False):
        """host: a C-contiguous array, whose bytes go to dev_ptr on `stream`.
        They have been read when this returns; the copy may still run.
        following: nothing but uploads has been queued there since one that
        waited for the stream."""
        slots = self.up if host.nbytes <= _SLOT * _SLOTS else self._big()
        slots.copy(_COPY_UP_NEXT if following else _COPY_UP, dev_ptr, host,
                   self._threads(host.nbytes), stream)

    def to_host(self, out, dev_ptr, stream=None):
        """out: a C-contiguous array, filled from dev_ptr behind the work
        queued on `stream`."""
        if out.nbytes > _SLOT * _SLOTS:
            self._big().copy(_COPY_DOWN, dev_ptr, out, self._threads(out.nbytes), stream)
            return
        _lib.check(_lib.load().ozk_copy_to_host(
            out.ctypes.data, dev_ptr, out.nbytes, self.down, self.size, self.flags,
            self.counts, self._threads(out.nbytes), stream))

    def release(self, h):
        self.up.release(h)
        if self.big is not None:
            self.big.release(h)
        for p in (self.down, self.flags):
            h.hipHostFree(p)
        h.hipFree(self.counts)


class _Pool:
    """Device blocks by size class: powers of two below 1 MiB, multiples of
    2 MiB above.  Released blocks are kept up to `keep` bytes in all."""

    def __init__(self, rt, keep=64 << 30):
        self.rt, self.keep, self.cached = rt, keep, 0
        self.free = {}
        self.lock = threading.Lock()

    @staticmethod
    def size_class(n):
        n = max(int(n), 256)
        if n < (1 << 20):
            return 1 << (n - 1).bit_length()
        return -(-n // (2 << 20)) * (2 << 20)

    def take(self, n):
        c = self.size_class(n)
        with self.lock:
            lst = self.free.get(c)
            if lst:
                self.cached -= c
                return lst.pop(), c
        return self.rt.malloc(c), c

    def give(self, ptr, c):
        with self.lock:
            if self.cached + c <= self.keep:
                self.free.setdefault(c, []).append(ptr)
                self.cached += c
                return
        self.rt.free(ptr)


class _Block:
    """One pool block, returned to the pool when the last array using it is
    collected.  Work that still reads it was queued on the null stream
    before any later use of the block, so reuse on the null stream stays in
    order; a user that writes a block on another stream first synchronizes
    the null stream (matmul's two-halves path does)."""
    __slots__ = ("ptr", "cls", "__weakref__")

    def __init__(self, nbytes):
        self.ptr, self.cls = _pool().take(nbytes)

    def __del__(self):
        try:
            _pool().give(self.ptr, self.cls)
        except Exception:  # interpreter shutdown
            pass


class DeviceArray:
    """A device array of the NumPy family: a 2-D array has C-ordered rows
    with `ld` elements from one row to the next; other ranks are contiguous."""

    def __init__(self, shape, dtype=np.float64, ld=None, block=None, offset=0):
        self.shape = tuple(int(s) for s in shape)
        self.dtype = np.dtype(dtype)
        if len(self.shape) == 2:
            rows, cols = self.shape
            self.ld = int(ld) if ld is not None else max(cols, 1)
            count = max(rows - 1, 0) * self.ld + cols if rows and cols else 0
        else:
            self.ld = None
            count = int(np.prod(self.shape)) if self.shape else 1
        self.nbytes = count * self.dtype.itemsize
        self._block = block if block is not None else _Block(max(self.nbytes, 1))
        self._offset = offset

    # the protocol the host layer uses (shared with torch tensors)
    def data_ptr(self):
        return self._block.ptr + self._offset

    def dim(self):
        return len(self.shape)

    @property
    def ndim(self):
        return len(self.shape)

    def numel(self):
        return int(np.prod(self.shape)) if self.shape else 1

    def stride(self, d):
        return (self.ld, 1)[d] if len(self.shape) == 2 else 1

    def element_size(self):
        return self.dtype.itemsize

    def column(self):
        """A 1-D array as its (n, 1) matrix (same memory)."""
        return DeviceArray((self.shape[0], 1), self.dtype, 1, self._block, self._offset)

    def flat(self):
        """An (n, 1) matrix as its 1-D array (same memory)."""
        return DeviceArray((self.shape[0],), self.dtype, None, self._block, self._offset)

    @classmethod
    def from_numpy(cls, a, place=ALONE):
        """place: FIRST of several uploads, or FOLLOWING others with nothing
        else queued since the first."""
        a = np.ascontiguousarray(a)
        d = cls(a.shape, a.dtype)
        assert d.nbytes == a.nbytes
        if a.nbytes >= (_ALONE_MIN if place == ALONE else _COPY_MIN):
            _stager().to_device(d.data_ptr(), a, following=place == FOLLOWING)
        else:
            _rt().copy(d.data_ptr(), a.ctypes.data, a.nbytes, _H2D)
        return d

    def numpy(self):
        """Synchronising copy to a new NumPy array."""
        out = np.empty(self.shape, self.dtype)
        if out.size == 0:
            return out
        if self.dim() == 2 and self.ld != self.shape[1]:
            full = np.empty((self.shape[0], self.ld), self.dtype)
            _rt().copy(full.ctypes.data, self.data_ptr(), self.nbytes, _D2H)
            out[:] = full[:, :self.shape[1]]
        elif out.nbytes >= _COPY_MIN:
            _stager().to_host(out, self.data_ptr())
        else:
            _rt().copy(out.ctypes.data, self.data_ptr(), out.nbytes, _D2H)
        return out

    @classmethod
    def zeros(cls, shape, dtype=np.float64):
        d = cls(shape, dtype)
        _rt().memset(d.data_ptr(), 0, d.nbytes)
        return d

    def copy_from(self, other):
        """Device-to-device copy of an array of the same shape and layout."""
        if other.shape != self.shape or other.nbytes != self.nbytes:
            raise ValueError("copy between arrays of different shape or layout")
        _rt().copy(self.data_ptr(), other.data_ptr(), self.nbytes, _D2D)


class _Blas:
    """rocBLAS FP64 products on the null stream.  Row-major matrices are
    column-major transposes, so C = A B is computed as C^T = B^T A^T."""

    def __init__(self):
        _rt()
        b = _open("librocblas.so.5")
        vp, i = ctypes.c_void_p, ctypes.c_int
        dp = ctypes.POINTER(ctypes.c_double)
        b.rocblas_create_handle.restype = i
        b.rocblas_create_handle.argtypes = [ctypes.POINTER(vp)]
        b.rocblas_set_stream.restype = i
        b.rocblas_set_stream.argtypes = [vp, vp]
        b.rocblas_dgemm.restype = i
        b.rocblas_dgemm.argtypes = [vp, i, i, i, i, i, dp, vp, i, vp, i, dp, vp, i]
        b.rocblas_dgeam.restype = i
        b.rocblas_dgeam.argtypes = [vp, i, i, i, i, dp, vp, i, dp, vp, i, vp, i]
        b.rocblas_destroy_handle.restype = i
        b.rocblas_destroy_handle.argtypes = [vp]
        h = vp()
        self._chk(b.rocblas_create_handle(ctypes.byref(h)), "rocblas_create_handle")
        self._chk(b.rocblas_set_stream(h, None), "rocblas_set_stream")
        self.b, self.h = b, h

    @staticmethod
    def _chk(rc, what):
        if rc != 0:
            raise _lib.OzakiError(f"{what} failed: rocblas status {rc}")

    @staticmethod
    def _c(x):
        return ctypes.byref(ctypes.c_double(x))

    def matmul(self, A, B, C, alpha=1.0, beta=0.0):
        """C = alpha A B + beta C (row-major A: N x K, B: K x M, C: N x M)."""
        N, K = A.shape
        M = B.shape[1]
        if N == 0 or M == 0:
            return C
        if K == 0:
            raise ValueError("contraction length 0")
        self._chk(self.b.rocblas_dgemm(self.h, _OP_N, _OP_N, M, N, K, self._c(alpha),
                                       B.data_ptr(), B.ld, A.data_ptr(), A.ld, self._c(beta),
                                       C.data_ptr(), C.ld), "rocblas_dgemm")
        return C

    def gram(self, A, G):
        """G = A^T A (row-major A: rows x cols, G: cols x cols)."""
        rows, cols = A.shape
        self._chk(self.b.rocblas_dgemm(self.h, _OP_N, _OP_T, cols, cols, rows, self._c(1.0),
                                       A.data_ptr(), A.ld, A.data_ptr(), A.ld, self._c(0.0),
                                       G.data_ptr(), G.ld), "rocblas_dgemm")
        return G

    def add(self, A, B, out):
        """out = A + B (row-major matrices of one shape; one rounding per
        element, as an FP64 add)."""
        n, m = A.shape
        if n and m:
            self._chk(self.b.rocblas_dgeam(self.h, _OP_N, _OP_N, m, n, self._c(1.0),
                                           A.data_ptr(), A.ld, self._c(1.0), B.data_ptr(),
                                           B.ld, out.data_ptr(), out.ld), "rocblas_dgeam")
        return out

    def half_sum_transpose(self, G, out):
        """out = G * 0.5 + G^T * 0.5, which equals (G + G^T) * 0.5 exactly
        (halving is exact, and one rounding of the same sum)."""
        n = G.shape[0]
        self._chk(self.b.rocblas_dgeam(self.h, _OP_N, _OP_T, n, n, self._c(0.5), G.data_ptr(),
                                       G.ld, self._c(0.5), G.data_ptr(), G.ld,
                                       out.data_ptr(), out.ld), "rocblas_dgeam")
        return out


_state = {}
# Re-entrant: a maker may create another singleton (the stager's and the
# pool's makers take the runtime), and any of them may be the first created.
_state_lock = threading.RLock()


def _get(name, make):
    v = _state.get(name)
    if v is None:
        with _state_lock:
            v = _state.get(name)
            if v is None:
                v = make()
                _state[name] = v
    return v


def _rt():
    return _get("rt", _Runtime)


_exit_hooks = []  # called with the runtime's entry points once the device is idle


def _release_at_exit():
    """At interpreter exit, before the runtime's own teardown: let queued
    work end, then release what this package holds in the runtime (the
    staging buffers and their events, the rocBLAS handle, the compute stream,
    the pool's cached blocks, and through _exit_hooks what other modules keep),
    so that none of it is left for the runtime's static destructors.  The
    runtime and the pool stay: blocks that arrays release later are freed at
    once.  Errors are ignored: the runtime may be unusable by then."""
    with _state_lock:
        st = dict(_state)
        for k in st:
            if k not in ("rt", "pool"):
                _state.pop(k, None)
    rt = st.get("rt")
    if rt is None:
        return
    h = rt.h
    try:
        h.hipDeviceSynchronize()
        for hook in _exit_hooks:
            hook(h)
        for stager in st.values():
            if isinstance(stager, _Stager):
                stager.release(h)
        blas_ = st.get("blas")
        if blas_ is not None:
            blas_.b.rocblas_destroy_handle(blas_.h)
        if st.get("cstream") is not None:
            h.hipStreamDestroy(st["cstream"])
        pool = st.get("pool")
        if pool is not None:
            with pool.lock:
                for ptrs in pool.free.values():
                    for ptr in ptrs:
                        h.hipFree(ptr)
                pool.free.clear()
                pool.cached = 0
                pool.keep = 0  # blocks released later are freed, not kept
        h.hipGetLastError()
    except Exception:
        pass


atexit.register(_release_at_exit)


def _pool():
    return _get("pool", lambda: _Pool(_rt()))


def _stager():
    """The current device's pinned memory for host copies."""
    return _get(("stager", _rt().device()), lambda: _Stager(_rt()))


def compute_stream():
    """The NumPy family's stream for work that overlaps its null-stream
    copies (kept for the process)."""
    return _get("cstream", lambda: _rt().nonblocking_stream())


def blas():
    return _get("blas", _Blas)


def device_count():
    return _rt().device_count()


def sync():
    _rt().sync()
