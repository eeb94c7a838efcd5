"""Device memory, streams and events for the Python host mirror (thin HIP runtime plumbing)."""
import ctypes as C
import threading

import numpy as np

from . import _lib
from ._lib import hip, hip_check


class DeviceBuffer:
    """Owning handle on a hipMalloc allocation."""

    def __init__(self, nbytes):
        self.nbytes = int(nbytes)
        p = C.c_void_p(0)
        hip_check(hip.hipMalloc(C.byref(p), max(self.nbytes, 4)), "hipMalloc(%d)" % self.nbytes)
        self.ptr = p.value

    @classmethod
    def from_numpy(cls, arr):
        arr = np.ascontiguousarray(arr)
        buf = cls(arr.nbytes)
        if arr.nbytes:
            hip_check(hip.hipMemcpy(buf.ptr, arr.ctypes.data, arr.nbytes, _lib.H2D), "hipMemcpy H2D")
        return buf

    @classmethod
    def zeros(cls, nbytes):
        buf = cls(nbytes)
        buf.fill(0)
        return buf

    def fill(self, byte):
        if self.nbytes:
            hip_check(hip.hipMemset(self.ptr, byte, self.nbytes), "hipMemset")

    def upload(self, arr):
        arr = np.ascontiguousarray(arr)
        assert arr.nbytes <= self.nbytes
        hip_check(hip.hipMemcpy(self.ptr, arr.ctypes.data, arr.nbytes, _lib.H2D), "hipMemcpy H2D")

    def to_numpy(self, dtype, shape):
        out = np.empty(shape, dtype=dtype)
        assert out.nbytes <= self.nbytes, (out.nbytes, self.nbytes)
        if out.nbytes:
            hip_check(hip.hipMemcpy(out.ctypes.data, self.ptr, out.nbytes, _lib.D2H), "hipMemcpy D2H")
        return out

    def free(self):
        if getattr(self, "ptr", None):
            hip.hipFree(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class PinnedBuffer:
    """Owning handle on pinned host memory."""

    def __init__(self, nbytes):
        self.nbytes = int(nbytes)
        p = C.c_void_p(0)
        hip_check(hip.hipHostMalloc(C.byref(p), max(self.nbytes, 4), 0), "hipHostMalloc(%d)" % self.nbytes)
        self.ptr = p.value
        self.bytes = np.ctypeslib.as_array((C.c_uint8 * self.nbytes).from_address(self.ptr))

    def free(self):
        if getattr(self, "ptr", None):
            self.bytes = None
            hip.hipHostFree(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class Downloads:
    """Results that are downloaded over and over: from the second time on through pinned memory (a copy to pageable memory
    takes 25 us where that takes 10), which the first result need not pay for, and without it where there is none to be
    had.  Downloads of one object take turns."""

    def __init__(self):
        self.lock = threading.Lock()
        self.count = 0
        self.pinned = None

    def get(self, src, dtype, shape):
        """A new array of the device buffer's first bytes."""
        with self.lock:
            self.count += 1
            if self.count == 2:
                try:
                    self.pinned = PinnedBuffer(src.nbytes)
                except _lib.TcbnnError:
                    hip.hipGetLastError()  # (reported here, not by the next launch)
            if self.pinned is None:
                return src.to_numpy(dtype, shape)
            out = np.empty(shape, dtype=dtype)
            assert out.nbytes <= min(self.pinned.nbytes, src.nbytes), (out.nbytes, self.pinned.nbytes, src.nbytes)
            if out.nbytes:
                hip_check(hip.hipMemcpy(self.pinned.ptr, src.ptr, out.nbytes, _lib.D2H), "hipMemcpy D2H")
                out.reshape(-1).view(np.uint8)[:] = self.pinned.bytes[:out.nbytes]
            return out

    def free(self):
        with self.lock:
            self.count = 0
            if self.pinned is not None:
                self.pinned.free()
                self.pinned = None


class Uploader:
    """Uploads of new input batches through pinned memory (tcbnn_upload)."""

    def __init__(self, nbytes, staged=False):
        p = C.c_void_p(0)
        _lib.check(_lib.lib.tcbnn_uploader_create(int(nbytes), int(staged), C.byref(p)))
        self.handle = p.value

    def upload(self, dst, arr):
        assert arr.nbytes <= dst.nbytes
        _lib.check(_lib.lib.tcbnn_upload(self.handle, dst.ptr, arr.ctypes.data, arr.nbytes))

    def stage(self, arr):
        """max |x| of the array, which commit() writes to its destination."""
        most = C.c_float(0)
        _lib.check(_lib.lib.tcbnn_upload_stage(self.handle, arr.ctypes.data, arr.size, C.byref(most)))
        return most.value

    def commit(self, dst):
        _lib.check(_lib.lib.tcbnn_upload_commit(self.handle, dst.ptr))

    def free(self):
        if getattr(self, "handle", None):
            _lib.lib.tcbnn_uploader_destroy(self.handle)
            self.handle = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class InputUploads:
    """New batches for a layer's input buffer.  put() is one call per batch, whichever threads they come from: the
    uploader keeps ONE staged batch, so what stages it, judges it and commits it must not be interleaved.  The first batch
    is scanned and copied as it is: an uploader costs more to make (4 ms for 38.5 MB) than it saves on one batch (1 ms).
    Where none can be made every batch goes that way."""

    def __init__(self, staged=False):
        self.staged = staged
        self.lock = threading.Lock()
        self.count = 0
        self.uploader = None

    def put(self, dst, x, accept=None):
        """Replaces the contents of `dst` by `x`.  accept(max |x|) (staged uploads) raises to refuse the batch; the
        buffer then keeps what it holds."""
        with self.lock:
            self.count += 1
            if self.count == 2:
                try:
                    self.uploader = Uploader(dst.nbytes, self.staged)
                except _lib.TcbnnError:
                    pass
            if self.uploader is None:
                if accept is not None:
                    accept(_lib.lib.tcbnn_host_abs_max(x.ctypes.data, x.size))
                dst.upload(x)
            elif accept is None:
                self.uploader.upload(dst, x)
            else:
                accept(self.uploader.stage(x))
                self.uploader.commit(dst)

    def free(self):
        with self.lock:
            self.count = 0
            if self.uploader is not None:
                self.uploader.free()
                self.uploader = None


class Stream:
    """A HIP stream at the default priority."""

    def __init__(self):
        p = C.c_void_p(0)
        hip_check(hip.hipStreamCreate(C.byref(p)), "hipStreamCreate")
        self.handle = p.value

    def synchronize(self):
        hip_check(hip.hipStreamSynchronize(self.handle), "hipStreamSynchronize")

    def __del__(self):
        try:
            if self.handle:
                hip.hipStreamDestroy(self.handle)
        except Exception:
            pass


class Event:
    def __init__(self):
        p = C.c_void_p(0)
        hip_check(hip.hipEventCreate(C.byref(p)), "hipEventCreate")
        self.handle = p.value

    def record(self, stream=None):
        hip_check(hip.hipEventRecord(self.handle, stream.handle if stream else None), "hipEventRecord")

    def synchronize(self):
        hip_check(hip.hipEventSynchronize(self.handle), "hipEventSynchronize")

    def elapsed_ms(self, end):
        ms = C.c_float(0)
        hip_check(hip.hipEventElapsedTime(C.byref(ms), self.handle, end.handle), "hipEventElapsedTime")
        return ms.value

    def __del__(self):
        try:
            if self.handle:
                hip.hipEventDestroy(self.handle)
        except Exception:
            pass


class Graph:
    """A HIP graph captured from the launches `record(stream)` makes on `stream` (the layers' forward
    calls allocate nothing and clear nothing with memset, so a whole network can be captured); replay
    with launch().  The caller warms the launches up once before capturing."""

    def __init__(self, stream, record):
        self.stream = stream
        g = C.c_void_p(0)
        hip_check(hip.hipStreamBeginCapture(stream.handle, 0), "hipStreamBeginCapture")  # global mode
        try:
            record(stream)
        finally:
            hip_check(hip.hipStreamEndCapture(stream.handle, C.byref(g)), "hipStreamEndCapture")
        self.graph = g.value
        e = C.c_void_p(0)
        hip_check(hip.hipGraphInstantiate(C.byref(e), self.graph, None, None, 0), "hipGraphInstantiate")
        self.exec = e.value

    def launch(self):
        hip_check(hip.hipGraphLaunch(self.exec, self.stream.handle), "hipGraphLaunch")

    def __del__(self):
        try:
            if getattr(self, "exec", None):
                hip.hipGraphExecDestroy(self.exec)
            if getattr(self, "graph", None):
                hip.hipGraphDestroy(self.graph)
        except Exception:
            pass

