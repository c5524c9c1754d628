"""The device backend over a stand-in for the library: its entry points as ctypes callbacks on host memory, a few of them computed
with numpy.  For the host side of a call -- recordings, calls laid out once, buffer ownership -- on a machine without a GPU.
`install()` goes before the first import of `nx_amd.backend`, so in a process of its own."""
import ctypes as C

import numpy as np

memory = {}      # handle -> its bytes
_spare = []      # handles given back: the next buffer takes the last one, as an allocator gives out an address again
_next = [1 << 20]
_error = [b""]
deferred = []    # what an earlier kernel recorded: the next waiting call reports it, once
counts = {}      # calls per entry point
refused = set()  # entry points that answer HIPNX_EUNSUPPORTED
DTYPES = [np.uint8, np.uint16, np.uint32, np.uint64, np.int8, np.int16, np.int32, np.int64, np.float16, None, np.float32, np.float64]


def _new(nbytes, fill=0xA5):
    handle = _spare.pop() if _spare else _next[0]
    if handle == _next[0]:
        _next[0] += 64
    memory[handle] = np.full(max(nbytes, 1), fill, np.uint8)
    return handle


def _view(handle, dt, n):
    return memory[handle].view(np.uint8)[:n * np.dtype(DTYPES[dt]).itemsize].view(DTYPES[dt])


def _raise_deferred():
    if not deferred:
        return 0
    _error[0] = deferred.pop()
    return 8  # HIPNX_ERAISED


def install():
    from nx_amd import _lib as L
    from nx_amd import backend_names as names

    def ctx_create(device, out):
        out[0] = 4096 + device
        return 0

    def buf_alloc(ctx, nbytes, out):
        out[0] = _new(nbytes)
        return 0

    def buf_destroy(handle):
        del memory[handle]
        _spare.append(handle)
        return 0

    def buf_wrap(ctx, address, nbytes, out):  # (an address here is the handle of the buffer that owns the memory)
        owned = memory[address]
        out[0] = _new(0)
        memory[out[0]] = owned
        return 0

    def fill(ctx, handle, size, src, n):
        memory[handle][:size * n] = np.tile(np.frombuffer(C.string_at(src, size), np.uint8), n)
        return 0

    def h2d(ctx, handle, at, src, n):
        memory[handle][at:at + n] = np.frombuffer(C.string_at(src, n), np.uint8)
        return 0

    def d2h(ctx, handle, at, dst, n):
        C.memmove(dst, memory[handle][at:at + n].tobytes(), n)
        return _raise_deferred()

    def d2d(ctx, dst, at, src, src_at, n):
        memory[dst][at:at + n] = memory[src][src_at:src_at + n]
        return 0

    def binary(ctx, op, lc, rc, oc, rank, dims, ls, rs, l, r, out):
        shape = [dims[i] for i in range(rank)]

        def operand(handle, code, strides):
            base = memory[handle].view(np.uint8)
            size = np.dtype(DTYPES[code]).itemsize
            return np.lib.stride_tricks.as_strided(base[:base.size // size * size].view(DTYPES[code]), shape, [strides[i] * size for i in range(rank)])
        a, b = operand(l, lc, ls), operand(r, rc, rs)
        name = names.BINARY_OPS[op]
        with np.errstate(all="ignore"):
            v = {"add": lambda: a + b, "subtract": lambda: a - b, "multiply": lambda: a * b, "divide": lambda: a / b,
                 "equal": lambda: a == b, "greater": lambda: a > b}[name]()
        memory[out][:v.size * np.dtype(DTYPES[oc]).itemsize] = np.ascontiguousarray(v).astype(DTYPES[oc]).ravel().view(np.uint8)
        return 0

    def unary(ctx, op, ic, oc, n, t, out):
        f = {"exp": np.exp, "negate": np.negative}[names.UNARY_OPS[op]]
        _view(out, oc, n)[:] = f(_view(t, ic, n))
        return 0

    def gather(ctx, elem, rank, dims, dt, n, depth, policy, t, idx, out):
        row = elem * int(np.prod([dims[i] for i in range(1, rank)]))
        at = _view(idx, dt, n)
        if policy == 0:  # waits for its kernel
            if ((at < 0) | (at >= dims[0])).any():
                _error[0] = b"index out of bounds"
                return 6
            if status := _raise_deferred():
                return status
        memory[out][:n * row] = memory[t][:dims[0] * row].reshape(dims[0], row)[np.clip(at, 0, dims[0] - 1)].ravel()
        return 0

    def last_error(dst, cap):
        C.memmove(dst, _error[0] + b"\0", len(_error[0]) + 1)
        return 0

    def ok(*args):
        return 0

    def unsupported(*args):
        _error[0] = b"not in the stand-in"
        return 7

    made = {"hipnx_ctx_create": ctx_create, "hipnx_buf_alloc": buf_alloc, "hipnx_buf_destroy": buf_destroy, "hipnx_buf_wrap": buf_wrap,
            "hipnx_buf_free": ok, "hipnx_buf_device_ptr": lambda handle: handle, "hipnx_fill": fill, "hipnx_h2d": h2d, "hipnx_d2h": d2h,
            "hipnx_d2d": d2d, "hipnx_binary": binary, "hipnx_unary": unary, "hipnx_last_error": last_error, "hipnx_fused_set_mode": ok,
            "hipnx_gather": gather, "hipnx_capture_begin": ok}

    class Library:
        pass
    lib = Library()
    for name, args in L.PROTOTYPES.items():
        def entry(*a, _fn=made.get(name, unsupported), _name=name):
            counts[_name] = counts.get(_name, 0) + 1
            return _fn(*a) if _name not in refused else unsupported()
        if name == "hipnx_last_error":  # (a char pointer arrives as bytes otherwise)
            args = [C.c_void_p, C.c_size_t]
        fn = C.CFUNCTYPE(C.c_void_p if name == "hipnx_buf_device_ptr" else C.c_int, *args)(entry)
        fn.argtypes = args
        setattr(lib, name, fn)
    L.lib = lib
