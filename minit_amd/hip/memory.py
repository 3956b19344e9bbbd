"""Device memory, streams and events over the C ABI.

``HIPMemory`` mirrors the reference's ``CUDAMemory`` (minit/cuda/allocator.py:
85-117: pointer + size, freed in ``__del__``, ``copy_from`` / ``copy`` /
``reset``).  The reference draws from ``cudaMallocAsync``'s pool; here freed
blocks go to a small size-keyed free list so a steady-state loop does not call
``hipMalloc`` / ``hipFree`` (which synchronises the device) per tensor.
"""
import ctypes
import threading
from collections import OrderedDict
from functools import lru_cache
from typing import Dict, List, Optional

from .. import lib

# Free blocks by their size, the sizes used last at the end.  What does not fit under the limit any more
# makes room by giving back the sizes that have gone unused for longest: a pool that keeps the first 4 GiB it
# sees sends every later size through hipMalloc and hipFree (attention over 32 heads of 1977 tokens after
# other lengths: 14.2 ms a pass, of which the kernels take 0.3).
_POOL: "OrderedDict[int, List[int]]" = OrderedDict()
_POOL_BYTES = 0
_POOL_LIMIT = 4 << 30
# Blocks handed out for less than their size: pointer -> size.
_LENT: Dict[int, int] = {}
# Reentrant: a tensor may die (and release its block) while the lock is held.  Whatever allocates a container
# may run the collector, so nothing read from the pool before such a place is relied on behind it.
_POOL_LOCK = threading.RLock()


def _round(size: int) -> int:
    """Block size for ``size`` bytes: a multiple of 256."""
    return (size + 255) // 256 * 256 if size > 256 else 256


def _malloc(size: int) -> int:
    ptr = ctypes.c_void_p()
    lib.call("mh_malloc", ctypes.byref(ptr), size)
    return ptr.value


def _take_larger(size: int) -> Optional[int]:
    """The smallest free block of up to an eighth more than ``size``: a prompt of another length finds the blocks of a
    longer one and not a hipMalloc each.  A new block has the size that was asked for, so that weights and
    caches take no more memory than they need."""
    global _POOL_BYTES
    found, most = 0, size + size // 8
    for block in list(_POOL):
        if size < block <= most and (not found or block < found) and _POOL[block]:
            found = block
    if not found:
        return None
    ptr = _POOL[found].pop()
    _POOL_BYTES -= found
    _LENT[ptr] = found
    return ptr


def allocate(size: int) -> int:
    """A block of at least ``size`` bytes; ``release(ptr, size)`` gives it back."""
    global _POOL_BYTES
    size = (size + 255) // 256 * 256 if size > 256 else 256   # _round
    with _POOL_LOCK:
        bucket = _POOL.get(size)
        if bucket:
            _POOL_BYTES -= size
            return bucket.pop()
        if size > 1 << 20:
            ptr = _take_larger(size)
            if ptr is not None:
                return ptr
    try:
        return _malloc(size)
    except lib.HipError:
        empty_cache()
        return _malloc(size)


def release(ptr: int, size: int) -> None:
    global _POOL_BYTES
    size = (size + 255) // 256 * 256 if size > 256 else 256   # _round
    with _POOL_LOCK:
        if _LENT:
            size = _LENT.pop(ptr, size)
        if _POOL_BYTES + size > _POOL_LIMIT:
            if size > _POOL_LIMIT:
                lib.call("mh_free", ptr)
                return
            _make_room(size)
        bucket = _POOL.get(size)
        if bucket is None:
            bucket = _POOL.setdefault(size, [])
        bucket.append(ptr)
        _POOL.move_to_end(size)
        _POOL_BYTES += size


def _make_room(size: int) -> None:
    global _POOL_BYTES
    while _POOL and _POOL_BYTES + size > _POOL_LIMIT:
        oldest = next(iter(_POOL))
        bucket = _POOL[oldest]
        if not bucket:
            del _POOL[oldest]
            continue
        ptr = bucket.pop()
        _POOL_BYTES -= oldest
        lib.call("mh_free", ptr)


def empty_cache() -> None:
    global _POOL_BYTES
    with _POOL_LOCK:
        while _POOL:
            size, bucket = _POOL.popitem()
            _POOL_BYTES -= size * len(bucket)
            for ptr in bucket:
                lib.call("mh_free", ptr)


def synchronize(stream=None) -> None:
    """``sync_cuda`` of the reference (allocator.py:44-46)."""
    if stream is None:
        lib.call("mh_device_synchronize")
    else:
        lib.call("mh_stream_synchronize", stream)


def copy(dst: int, src: int, size: int, stream=None) -> None:
    lib.call("mh_memcpy", dst, src, size, stream)


class HIPMemory:
    __slots__ = ["_pointer", "_size", "_owner"]

    def __init__(self, size: int, pointer: int = None, owner=None) -> None:
        """Allocates ``size`` bytes, or wraps ``pointer`` kept alive by ``owner``."""
        self._size = size
        self._owner = owner
        self._pointer = allocate(size) if pointer is None else pointer

    def __del__(self):
        try:
            if self._owner is None and self._pointer is not None:
                release(self._pointer, self._size)
        except Exception:
            pass
        self._pointer = None

    def copy_from(self, src: "HIPMemory"):
        assert self._size == src._size
        copy(self._pointer, src._pointer, self._size)

    def copy(self) -> "HIPMemory":
        new = HIPMemory(self._size)
        copy(new._pointer, self._pointer, self._size)
        return new

    def reset(self):
        lib.call("mh_memset", self._pointer, 0, self._size, None)


class Event:
    """HIP event for timing work on a given stream."""

    def __init__(self):
        h = ctypes.c_void_p()
        lib.call("mh_event_create", ctypes.byref(h))
        self.handle = h.value

    def record(self, stream=None):
        lib.call("mh_event_record", self.handle, stream)

    def synchronize(self):
        lib.call("mh_event_synchronize", self.handle)

    def elapsed_ms(self, stop: "Event") -> float:
        ms = ctypes.c_float(0)
        lib.call("mh_event_elapsed_ms", ctypes.byref(ms), self.handle, stop.handle)
        return ms.value

    def __del__(self):
        try:
            lib.call("mh_event_destroy", self.handle)
        except Exception:
            pass


def create_stream() -> int:
    h = ctypes.c_void_p()
    lib.call("mh_stream_create", ctypes.byref(h))
    return h.value


_WORKSPACE = None
_OWNER_THREAD = None


def _single_thread(what: str) -> None:
    """The operator API is the reference's: one host thread, every launch on the null stream
    (minit/cuda/dispatch.py passes ``None`` for the stream throughout).  The free list above
    recycles a block as soon as its tensor dies and the workspace below is shared by every
    split-K launch; both are only safe while launches are ordered on one stream by one thread,
    so a second thread is refused instead of silently racing on partial sums."""
    global _OWNER_THREAD
    me = threading.get_ident()
    if _OWNER_THREAD is None:
        _OWNER_THREAD = me
    elif _OWNER_THREAD != me:
        raise lib.HipError(f"{what}: the operator API is single-threaded (null stream); callers with their own "
                           "threads or streams pass their own workspace to the C ABI")


def workspace(nbytes: int) -> HIPMemory:
    """Zero-initialised scratch shared by the split-K kernels of the null stream.

    The kernels leave the part that must be zero (their arrival counters) zeroed,
    so the buffer is cleared only when it is (re)allocated.
    """
    global _WORKSPACE
    if _OWNER_THREAD != threading.get_ident():
        _single_thread("memory.workspace")
    if _WORKSPACE is None or _WORKSPACE._size < nbytes:
        size = max(_round(nbytes), 64 << 20)
        synchronize()
        _WORKSPACE = HIPMemory(size)
        _WORKSPACE.reset()
        synchronize()
    return _WORKSPACE


# What a product needs depends on its sizes, on what the process was started with and, up to 32 rows of at most one column
# tile per CU, on MH_GEMM_SMALL_KW, which is read at every call: there it is below 20 MB at any setting, less than
# the shared workspace has at least.
@lru_cache(maxsize=4096)
def _product_bytes(m: int, n: int, k: int, group_size: int, bits: int) -> int:
    return max(lib.call("mh_gptq_workspace_bytes", m, n, k, group_size, bits), 256)


def product_workspace(m: int, n: int, k: int, group_size: int, bits: int) -> HIPMemory:
    """The workspace of the null stream, large enough for a quantized product of these sizes."""
    return workspace(_product_bytes(m, n, k, group_size, bits))
