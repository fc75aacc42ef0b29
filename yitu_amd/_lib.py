"""ctypes binding of libyitu_hip.so and the small amount of torch plumbing
(device pointers, current stream, cached workspace) shared by the op modules.

There is no CPU fallback: if the library is missing or a tensor is not on a HIP
device the call raises.
"""
import ctypes
import os
import threading
import weakref

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libyitu_hip.so")
_lib = None
_lock = threading.Lock()
# The C ABI these bindings were written for (yitu_abi_version() of include/yitu_hip.h). A
# library of another version has other argument lists: calling it would hand the kernels
# shifted pointers, so it is refused at load time.
ABI_VERSION = 4

c_i64 = ctypes.c_int64
c_int = ctypes.c_int
c_f32 = ctypes.c_float
c_size = ctypes.c_size_t
c_ptr = ctypes.c_void_p


def lib():
    """Loads the HIP library; raises if it has not been built."""
    global _lib
    if _lib is None:
        with _lock:
            if _lib is None:
                if not os.path.exists(LIB_PATH):
                    raise RuntimeError(
                        "libyitu_hip.so is not built; run `python -m yitu_amd.build` "
                        "(there is no CPU fallback)")
                l = ctypes.CDLL(LIB_PATH)
                l.yitu_abi_version.restype = ctypes.c_int
                found = l.yitu_abi_version()
                if found != ABI_VERSION:
                    raise RuntimeError(
                        "libyitu_hip.so has ABI version %d, these bindings need %d; rebuild it "
                        "with `python -m yitu_amd.build --force`" % (found, ABI_VERSION))
                l.yitu_last_error.restype = ctypes.c_char_p
                _lib = l
    return _lib


_ops = None


def ops():
    """The native side of the op modules (csrc/bind): checks, allocation, per-graph state and
    autograd nodes over the same library; raises if it has not been built."""
    global _ops
    if _ops is None:
        lib()  # present, and of the version these bindings were written for
        try:
            from . import _ops as native
        except ImportError as exc:
            raise RuntimeError("yitu_amd/_ops.so is not built; run `python -m yitu_amd.build` "
                               "(there is no CPU fallback): %s" % exc) from exc
        _ops = native
    return _ops


def check(rc, what):
    if rc != 0:
        msg = lib().yitu_last_error().decode("utf-8", "replace")
        raise RuntimeError("%s failed (code %d): %s" % (what, rc, msg))


def ptr(t):
    """Device address of a tensor (None -> NULL)."""
    if t is None:
        return c_ptr(0)
    return c_ptr(t.data_ptr())


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_ptr(device):
    """The current HIP stream of ``device`` as a pointer argument."""
    if _raw_stream is not None and device.index is not None:
        return c_ptr(_raw_stream(device.index))  # no Stream object on the way
    return c_ptr(torch.cuda.current_stream(device).cuda_stream)


def require_device(*tensors):
    dev = None
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("expected a tensor on the GPU (HIP device), got %s" % t.device)
        if not t.is_contiguous():
            raise RuntimeError("expected a contiguous tensor")
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise RuntimeError("tensors live on different devices: %s vs %s" % (dev, t.device))
    return dev


def require_dtype(t, dtype, name):
    if t.dtype != dtype:
        raise RuntimeError("%s must be %s, got %s" % (name, dtype, t.dtype))


def workspace(n_bytes, device):
    """Scratch buffer for one call; the caching allocator makes this cheap and
    stream-ordered reuse keeps concurrent ops on one stream from colliding."""
    n = max(int(n_bytes), 256)
    return torch.empty(n, dtype=torch.uint8, device=device)


# ---- state derived from a graph ----------------------------------------------------
# The widest row, the row plan, the by-source view and by-source weight copies are
# functions of the index tensors and are kept per tensor OBJECT (implementation, address,
# version counter) for as long as the tensor lives (csrc/bind/graph_state.cpp). The version counter moves when torch writes
# the tensor; it does NOT move when a buffer is refilled through its raw pointer, which is
# how every kernel of this library (yitu_coo_to_csr, the device sampler, ...), DLPack
# consumers and foreign extensions write. Whoever refills an index or weight tensor in
# place must call ``forget`` on it (graph_ext.forget also drops the by-source state);
# the builders in data/csr.py and the samplers return fresh tensors and need not.
#
# Derived buffers are built on the stream that was current at the time; a later use on
# another stream waits for the build through an event recorded right behind it, and the
# buffers are not handed to anybody else before that use is over.


class _Built:
    __slots__ = ("value", "event", "raw_stream")

    def __init__(self, value, device):
        self.value = value
        self.raw_stream = stream_ptr(device).value
        self.event = torch.cuda.Event()
        self.event.record(torch.cuda.current_stream(device))

    def get(self, device):
        if stream_ptr(device).value != self.raw_stream:  # two integers in the common case
            stream = torch.cuda.current_stream(device)
            stream.wait_event(self.event)
            held = [self.value] if torch.is_tensor(self.value) else \
                [getattr(self.value, name) for name in self.value.__slots__]
            for t in held:
                if torch.is_tensor(t) and t.is_cuda:
                    t.record_stream(stream)
        return self.value


def watch(tensor):
    """Drops what is kept for ``tensor`` (csrc/bind/graph_state.cpp) when it dies."""
    native = ops()
    weakref.finalize(tensor, native.drop, native.impl_of(tensor)).atexit = False


_forgotten = {}  # id of a live tensor -> how often it was named to forget()


def forget(*tensors):
    """Drops every cached widest row and row plan derived from the given index tensors
    (call after refilling one of them in place through a raw pointer)."""
    for t in tensors:
        if t is not None:
            ops().drop(ops().impl_of(t))
            if id(t) not in _forgotten:
                weakref.finalize(t, _forgotten.pop, id(t), None).atexit = False
            _forgotten[id(t)] = _forgotten.get(id(t), 0) + 1


def state_of(tensors):
    """What changes when one of the tensors (which the caller keeps alive) is replaced, written
    by torch, or named to ``forget``: for copies kept beside what they were made from."""
    state = ops().tensor_state(tensors)
    return (state, [_forgotten.get(id(t), 0) for t in tensors]) if _forgotten else state


def max_degree(indptr):
    """Longest row of a CSR, computed once per ``indptr`` tensor (the kernels skip their
    hub-row machinery when no row reaches the hub threshold). The entry lives as long as the
    tensor object: an address alone is no identity, the allocator hands a freed block to the
    next graph of the same size."""
    native = ops()
    v = native.find_max_degree(indptr)
    if v < 0:
        if indptr.numel() <= 1:
            v = 0
        elif indptr.is_cuda and indptr.dtype == torch.int32 and indptr.dim() == 1 and \
                indptr.is_contiguous():
            v = int(native.longest_row(indptr).item())
        else:
            v = int((indptr[1:] - indptr[:-1]).max().item())
        put_max_degree(indptr, v)
    return v


def put_max_degree(indptr, value):
    """Keeps the longest row of a CSR whose builder knows it."""
    ops().put_max_degree(indptr, value)
    watch(indptr)


def row_plan(indptr, indices, n_src, col_mask):
    """Device buffer holding the row plan of (indptr, indices): band-ordered items of the long
    rows, a function of the graph only, built on the device on first use and kept while the
    index tensor lives. None when no row reaches the planning threshold and the graph is
    small. A larger graph without long rows gets the plan's header: it tells the row kernels
    whether most sources of a row lie near the row's own id, which decides how rows are dealt
    to the XCDs."""
    longest = max_degree(indptr)
    if longest < 64 and indices.numel() < ops().plan_min_edges:
        return None
    native = ops()
    plan = native.find_plan(indptr, indices, int(n_src), col_mask)
    if plan is None:
        plan = native.build_plan(indptr, indices, int(n_src), col_mask, longest)
        native.put_plan(indptr, indices, int(n_src), col_mask, _Built(plan, indices.device))
        watch(indices)
    return plan


def size_fn(name):
    fn = getattr(lib(), name)
    fn.restype = c_size
    return fn
