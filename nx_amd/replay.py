"""A traced function's library calls, recorded once and issued again without the evaluator.

The evaluator walks the graph on every call: 5-7 us of Python per node beside the 4 us of the library.  What it ends up
calling -- which entry points, with which extents, on which buffers, allocated and released in which order -- follows from
the traced shapes and types alone unless a node looks at values (`while`, `cond`) or moves data between host and device.
So one evaluation is recorded at the boundary of the library (every call through `_lib.lib`, every buffer made and
released), and later calls issue the same list natively (`csrc/calls.c`) on that call's own operands and fresh buffers:
no result and no address is kept.  A recording holds for the settings it was made under, kept for when they come back; whatever
it does not cover -- operands elsewhere, a device that is capturing, a call the library refuses -- is evaluated as before.
"""
from __future__ import annotations

import ctypes as C
import threading

from . import _lib as L
from . import backend as B
from . import nx as Nx
from ._lib import native

# entry points whose effect is their result buffer's content, a function of their arguments
_RECORDED = frozenset("hipnx_" + n for n in (
    "binary", "unary", "as_type", "reduce", "argreduce", "dot", "dot_strided", "dot_scaled", "dot_scaled_any_k", "transpose", "broadcast", "gather", "select", "clip",
    "concat", "strided_copy", "iota", "eye", "narrow_int", "threefry2x32", "threefry_key", "fused_elementwise", "fused_words", "fused_words_key", "fused_scores"))
_lock = threading.Lock()


class _Unrecordable(Exception):
    pass


class _Recorder:
    """Stands in for the library while one thread's evaluation is recorded (other threads pass through)."""

    def __init__(self, device, params):
        self._lib, self._thread = L.lib, threading.get_ident()
        self.ctx, self.device = B._Context.get(device), device
        self.slots, self.n_slots = {}, 0  # handle -> slot while the buffer lives
        self.ops, self.keep, self.freed, self.modes = [], [], [], set()
        self.failed, self.settings = False, B.settings()
        self.shapes = tuple((p.type, p.shape) for p in params)
        for p in params:
            self._slot(p.data.ref.handle)
        self.n_params = self.n_slots
        self.late = []  # handles of buffers made before the recording (constants): slots behind the parameters

    def _slot(self, handle):
        self.slots[handle] = self.n_slots
        self.n_slots += 1
        return self.n_slots - 1

    def __getattr__(self, name):
        real = getattr(self._lib, name)
        if threading.get_ident() != self._thread or not callable(real):
            return real

        def call(*args):
            status = real(*args)
            if self.failed or name in ("hipnx_fused_set_mode", "hipnx_last_error"):  # (a refusal is asked for its reason)
                return status
            if name not in _RECORDED:
                self.failed = True
            elif status == L.OK:
                try:
                    self._drain()
                    self.ops.append(("call", C.cast(real, C.c_void_p).value, [self._argument(a, t) for a, t in zip(args, real.argtypes)]))
                    if name in ("hipnx_fused_elementwise", "hipnx_fused_words", "hipnx_fused_words_key", "hipnx_fused_scores"):
                        self.modes.add(B._fused_set.get(self.device, "interpreted"))
                except Exception:  # the evaluation goes on, whatever becomes of its recording
                    self.failed = True
            return status
        return call

    def unrecordable(self):
        self.failed |= threading.get_ident() == self._thread

    def allocated(self, ref):
        if threading.get_ident() == self._thread:
            self._drain()
            self.ops.append(("alloc", self._slot(ref.handle), ref.nbytes))

    def _drain(self):
        """What has been released since the last call, in order."""
        for handle in self.freed:
            slot = self.slots.pop(handle, None)
            if slot is not None:
                self.ops.append(("free", slot))
        self.freed.clear()

    def _buffer(self, handle):
        slot = self.slots.get(handle)
        if slot is None:  # a constant the backend keeps: an operand of every call from now on
            ref = next((r for r in B.HipNxBackend._scalar_cache.copy().values() if r.handle == handle), None)  # (other threads add to it)
            if ref is None:
                raise _Unrecordable
            slot = self._slot(handle)
            self.late.append((slot, ref))
        return slot

    def _argument(self, a, argtype):
        if isinstance(a, C.c_void_p):
            self.keep.append(a)
            return a.value or 0
        if a is None:
            return 0
        if isinstance(a, int):
            return ("slot", self._buffer(a)) if argtype is C.c_void_p else a
        if isinstance(a, C.Array):
            if a._type_ is C.c_void_p:
                return ("list", [self._buffer(h) for h in a if h])
            self.keep.append(a)
            return C.addressof(a)
        raise _Unrecordable


class Replay:
    """A recorded evaluation: `run(params)` gives its results, or None where it does not apply (to tensors of other types and
    shapes, or to what is no tensor, too)."""

    def __init__(self, calls, device, mode, constants, settings):
        self.calls, self.device, self.mode, self.constants = calls, device, mode, constants
        self.settings, self.backend = settings, Nx.default_backend()

    def run(self, params):
        if B._capturing or self.settings != B.settings():
            return None
        backend = Nx.default_backend()
        if backend is not self.backend and (backend[0] is not self.backend[0] or backend[1] != self.backend[1]):
            return None
        if self.mode is not None and B._fused_set.get(self.device, "interpreted") != self.mode:
            B._set_fused_mode(self.mode, self.device)
        return self.calls(*params, *self.constants)


RECORD_AT = 3   # by the third evaluation every program is compiled and every fallback has been found
ATTEMPTS = 3     # a function whose calls cannot be written down is not tried for ever
SETTINGS = 8     # settings whose recordings a function keeps


class _History:
    """A function's evaluations on the device under one value of the settings."""

    __slots__ = ("calls", "attempts", "replay")

    def __init__(self):
        self.calls = self.attempts = 0
        self.replay = None


def evaluate(compiled, params):
    """An evaluation of `compiled` on operands of the device backend that its present recording, if any, did not answer: by the
    recording of the present settings, or the general way, writing it down if it is time to."""
    if B._capturing:
        return compiled._walk(params)
    mod, opts = Nx.default_backend()
    key = (B.settings(), mod, repr(opts))
    known = compiled.recordings.get(key)
    if known is None:
        if len(compiled.recordings) >= SETTINGS:
            compiled.recordings.clear()
        known = compiled.recordings.setdefault(key, _History())
    if known.replay is not None:
        if known.replay is not compiled.replay:  # these settings were in force before
            compiled.replay = known.replay
            results = known.replay.run(params)
            if results is not None:
                return results
        return compiled._walk(params)
    known.calls += 1
    if known.calls >= RECORD_AT and known.attempts < ATTEMPTS and _recordable(params) and _lock.acquire(blocking=False):
        try:
            results, replay = record(compiled._walk, params)
            known.attempts += 1
        finally:
            _lock.release()
        if replay is not None:
            compiled.replay = known.replay = replay
        return results
    return compiled._walk(params)


def _recordable(params):
    """Whether an evaluation on these operands can be told apart by its calls.  (One buffer twice: which of the two a call reads
    cannot be.)"""
    data = [p.data for p in params]
    return bool(data) and not any(d.released or d.device != data[0].device for d in data) and len({id(d.ref) for d in data}) == len(data)


def record(evaluate, params):
    """(the results of `evaluate(params)`, a Replay of it or None).  One thread at a time."""
    device = params[0].data.device
    private = [_private(p) for p in params]
    recorder = _Recorder(device, private)
    real, L.lib, B._recorder[0] = L.lib, recorder, recorder
    native.log_freed(recorder.freed)
    try:
        results = evaluate(private)
    finally:
        native.log_freed(None)
        L.lib, B._recorder[0] = real, None
    replay = None if recorder.failed else _finish(recorder, results)
    return [_callers(t, private, params) for t in results], replay

def _private(p):
    """The parameter in a buffer that the function cannot know as its own: a call's operands are told apart by their handles, and
    a number given as an argument and the same number written in the function are one shared constant (of one element)."""
    return B.HipNxBackend.backend_copy(p, B.HipNxBackend, {"device": p.data.device}) if p.data.ref.nbytes <= 8 else p


def _callers(t, private, params):
    """A result that is a parameter, or shares its buffer, over the caller's own."""
    for q, p in zip(private, params):
        if q is p:
            continue
        if t.data is q.data:
            return t.with_(data=p.data)
        if getattr(t.data, "ref", None) is q.data.ref:
            p.data.ref.sharers += 1
            return t.with_(data=B.HipNxBackend(p.data.ref, p.data.device))
    return t


def _finish(rec, results):
    rec._drain()
    outs = []
    for t in results:
        d = t.data
        if d.__class__ is not B.HipNxBackend or d.device != rec.device:
            return None
        outs.append((rec.slots.get(d.ref.handle, -1), d.ref.nbytes, t.type, t.shape, t.names))
    late = [slot for slot, _ in rec.late]
    if rec.settings is not B.settings() or len(rec.modes) > 1 or len({o[0] for o in outs}) < len(outs) or any(o[0] < rec.n_params or o[0] in late for o in outs):
        return None  # (a parameter or a constant handed through, or one buffer under two results; settings that another thread changed meanwhile)
    # slots in the order the native side wants them: parameters, constants, then what is allocated
    order = list(range(rec.n_params)) + late + [s for s in range(rec.n_params, rec.n_slots) if s not in late]
    to = {s: i for i, s in enumerate(order)}

    def moved(a):
        if a.__class__ is not tuple:
            return a
        return (a[0], [to[s] for s in a[1]] if a[0] == "list" else to[a[1]])
    ops = [(op[0], op[1], [moved(a) for a in op[2]]) if op[0] == "call" else (op[0], to[op[1]], op[2] if op[0] == "alloc" else 0) for op in rec.ops]
    calls = native.record(ops, rec.n_params + len(late), rec.n_slots, [(to[o[0]],) + o[1:] for o in outs], rec.ctx, rec.ctx.value, rec.device, rec.keep, rec.shapes)
    constants = [Nx.Tensor(B.HipNxBackend(ref, rec.device), "u8", ()) for _, ref in rec.late]
    return Replay(calls, rec.device, rec.modes.pop() if rec.modes else None, constants, rec.settings)
