"""Traced functions and callbacks issued natively (nx_amd/replay.py, csrc/calls.c), over the stand-in for the library: one case per
function, run by name in a process of its own (test_recording.py)."""
import sys

import library_standin as standin

standin.install()

import numpy as np  # noqa: E402

from nx_amd import HostBinary, HipNxBackend as Hip  # noqa: E402
from nx_amd import backend as B  # noqa: E402
from nx_amd import defn  # noqa: E402
from nx_amd import nx as Nx  # noqa: E402
from support import from_numpy  # noqa: E402

Nx.default_backend(Hip)
FUSE = (False, True, "compiled")


def f32(*values):
    return from_numpy(np.asarray(values, np.float32), "f32", Hip)


def read(t):
    return Nx.to_numpy(t).tolist()


def a_number_given_as_an_argument_is_not_the_functions_own():
    """The number that is an argument when the recording is made is also written in the function."""
    for fuse in FUSE:
        x = f32(1, 2, 4)
        f = defn.compile(lambda x, s: (Nx.multiply(x, s), Nx.add(x, 0.5)), x, 0.5, fuse=fuse)
        for _ in range(4):
            f(x, 0.5)
        assert f.replay is not None
        scaled, shifted = f(x, 2.0)
        assert read(scaled) == [2, 4, 8] and read(shifted) == [1.5, 2.5, 4.5], (fuse, read(scaled), read(shifted))


def a_tensor_of_a_blocks_own_given_as_the_functions_argument():
    """A block's default function reads a tensor that the traced function is called with."""
    w, x = f32(1, 2, 4), f32(10, 20, 40)
    f = defn.compile(lambda v: Nx.block(object(), [v], v.with_(data=None), lambda struct, t: Nx.negate(w)), w)
    for _ in range(5):
        assert read(f(w)) == [-1, -2, -4]
    assert read(f(x)) == [-1, -2, -4]


def arguments_handed_through_stay_the_callers():
    x = f32(1, 2, 4)
    f = defn.compile(lambda v: (v, Nx.reshape(v, (3, 1)), Nx.multiply(v, 3.0)), x)
    for i in range(6):
        x = f32(i, 2, 4)
        same, alias, tripled = f(x)
        assert same.data is x.data and alias.data.ref is x.data.ref and read(tripled) == [3 * i, 6, 12]
        before = x.data.ref.sharers
        assert Nx.backend_deallocate(alias) == "ok" and x.data.ref.sharers == before - 1
        assert read(same) == [i, 2, 4]
    f = defn.compile(lambda s, v: (s, Nx.reshape(s, (1,)), Nx.multiply(v, s)), 2.0, x)
    for i in range(6):
        s = f32(3.0 + i) if i % 2 else Nx.to_tensor(2.0)
        s = Nx.reshape(s, ())
        same, alias, scaled = f(s, x)
        assert same.data is s.data and alias.data.ref is s.data.ref and alias.shape == (1,) and read(scaled) == [read(s) * v for v in read(x)]


def raises(call, text):
    try:
        call()
    except Exception as e:  # noqa: BLE001
        assert text in str(e), e
    else:
        raise AssertionError(f"no error, where {text!r} was due")


def what_an_earlier_kernel_recorded_is_raised_by_the_call_that_waits():
    """The library reports it once, to whichever call waits first: a callback laid out or recorded raises it, as any other does."""
    t, at = f32([1, 2], [3, 4], [5, 6]), from_numpy(np.array([2, 0], np.int32), "s32", Hip)
    f = defn.compile(lambda t, i: Nx.add(Nx.take(t, i), 1.0), t, at)
    for _ in range(5):
        assert read(Nx.take(t, at)) == [[5, 6], [1, 2]] and read(f(t, at)) == [[6, 7], [2, 3]]
    assert f.replay is not None
    for call in (lambda: Nx.take(t, at), lambda: f(t, at)):
        standin.deferred.append(b"ArithmeticError: divided by zero a while ago")
        raises(call, "divided by zero a while ago")
        assert not standin.deferred
        call()
    far = from_numpy(np.array([2, 3], np.int32), "s32", Hip)
    for call in (lambda: Nx.take(t, far), lambda: f(t, far)):
        raises(call, "index out of bounds")


def a_block_evaluated_by_its_default_function_while_a_recording_is_made():
    """Its callbacks come through the front end, which lays their calls out: after a setting changed, or after operands elsewhere."""
    for first in ("settings", "host"):
        x = f32(0, 2, 0)
        f = defn.compile(lambda a: Nx.logical_not(a), x)
        for i in range(6):
            if i == 2:
                previous = B.bounds_policy("clamp")
            here = x if first == "settings" or i > 1 else Nx.backend_copy(x, HostBinary, {})
            assert read(f(here)) == [1, 0, 1], (first, i)
        B.bounds_policy(previous)


def other_threads_make_constants_while_a_function_is_recorded():
    """The recorder looks its constants up in a table that grows meanwhile, and other threads' buffers are made while it begins and
    ends."""
    class Growing(dict):
        def values(self):
            for v in super().values():
                yield v
                self[len(self)] = v
    x = f32(1, 2, 4)
    f = defn.compile(lambda v: Nx.multiply(Nx.add(v, 0.25), 3.0), x)
    cache, Hip._scalar_cache = Hip._scalar_cache, Growing(Hip._scalar_cache)
    read(Nx.add(x, 7.0))
    try:
        for _ in range(5):
            assert read(f(x)) == [3.75, 6.75, 12.75]
    finally:
        Hip._scalar_cache = cache

    class Ending(list):  # (another thread ends its recording between two reads)
        def __getitem__(self, i):
            now, self[0] = list.__getitem__(self, i), None
            return now

    class Other:
        def allocated(self, ref):
            pass
    B._recorder = Ending([Other()])
    assert read(Nx.negate(x)) == [-1, -2, -4]
    B._recorder = [None]


def a_setting_changed_while_a_call_is_laid_out_or_recorded():
    """Another thread changes the bounds policy between the call's layout and its place in the table, or within the evaluation that
    is recorded: neither is kept under the new policy."""
    t, near, far = f32([1, 2], [3, 4], [5, 6]), from_numpy(np.array([2, 0], np.int32), "s32", Hip), from_numpy(np.array([2, 9], np.int32), "s32", Hip)
    prepared, armed = Hip.prepared.__func__, [1]

    def slowly(cls, *args):
        call = prepared(cls, *args)
        if armed:
            armed.clear()
            B.bounds_policy("clamp")
        return call
    Hip.prepared = classmethod(slowly)
    Nx.take(t, near)
    Hip.prepared = classmethod(prepared)
    assert read(Nx.take(t, far)) == [[5, 6], [5, 6]]
    f, evaluations = defn.compile(lambda t, i: Nx.take(t, i), t, near), []
    walk = f._walk

    def changing(params):
        evaluations.append(params)
        results = walk(params)
        if len(evaluations) == 3:
            B.bounds_policy("raise")
        return results
    f._walk = changing
    for _ in range(3):
        f(t, near)
    raises(lambda: f(t, far), "index out of bounds")


def recorded(f):
    """Whether a call of `f` is answered by its recording: nothing is evaluated."""
    walk, evaluated = f._walk, []
    f._walk = lambda params: (evaluated.append(1), walk(params))[1]
    try:
        yield lambda *args: (evaluated.clear(), f(*args), not evaluated)[2]
    finally:
        f._walk = walk


def recordings_are_made_again_and_come_back_with_their_settings():
    x, y = f32(1, 2, 4), f32(3, 5, 7)
    f = defn.compile(lambda a, b: Nx.subtract(Nx.multiply(a, 2.0), b), x, y)
    for by_recording in recorded(f):
        assert [by_recording(x, y) for _ in range(5)] == [False, False, False, True, True]
        B.bounds_policy("clamp")
        assert [by_recording(x, y) for _ in range(5)] == [False, False, False, True, True]
        B.bounds_policy("raise")     # back: the recording of these settings applies at once
        assert by_recording(x, y)
        B.bounds_policy("clamp")
        assert by_recording(x, y)
        Nx.default_backend(HostBinary)
        assert [by_recording(x, y) for _ in range(4)] == [False, False, False, True]
        Nx.default_backend(Hip)
        assert by_recording(x, y) and read(f(x, y)) == [-1, -1, 1]
        B.bounds_policy("raise")
        for i in range(20):          # any number of settings, a bounded number of recordings
            B.fused_mode("compiled", device=i)
            f(x, y)
            assert len(f.recordings) <= 8
        for i in range(20):
            B.fused_mode("interpreted", device=i)


def a_third_call_that_cannot_be_recorded_is_not_the_last_chance():
    import threading
    from nx_amd import replay
    x, y = f32(1, 2, 4), f32(3, 5, 7)
    host = Nx.backend_copy(x, HostBinary, {})
    f = defn.compile(lambda a, b: Nx.subtract(Nx.multiply(a, 2.0), b), x, y)
    for by_recording in recorded(f):
        assert not any(by_recording(x, x) for _ in range(4)) and f.replay is None  # one buffer twice
        assert not by_recording(x, y) and by_recording(x, y)
    f = defn.compile(lambda a, b: Nx.subtract(Nx.multiply(a, 2.0), b), x, y)
    for by_recording in recorded(f):
        assert not any(by_recording(host, y) for _ in range(4))                    # operands elsewhere count for nothing
        assert [by_recording(x, y) for _ in range(4)] == [False, False, False, True]
    f = defn.compile(lambda a, b: Nx.subtract(Nx.multiply(a, 2.0), b), x, y)
    for by_recording in recorded(f):
        assert not by_recording(x, y) and not by_recording(x, y)
        with replay._lock:                                                          # another thread records
            assert not by_recording(x, y)
        assert not by_recording(x, y) and by_recording(x, y)
    f = defn.compile(lambda a: Nx.logical_not(a), x)                                # never: tried a few times
    attempts, record = [], replay.record
    replay.record = lambda *a: (attempts.append(1), record(*a))[1]
    for _ in range(12):
        assert read(f(x)) == [0, 0, 0]
    replay.record = record
    assert f.replay is None and len(attempts) == replay.ATTEMPTS
    # two threads at once: whoever does not record leaves the other's recording alone
    f = defn.compile(lambda a, b: Nx.subtract(Nx.multiply(a, 2.0), b), x, y)
    threads = [threading.Thread(target=lambda: [f(x, y) for _ in range(50)]) for _ in range(4)]
    [t.start() for t in threads], [t.join() for t in threads]
    Nx.default_backend(Hip)
    for _ in range(3):
        assert read(f(x, y)) == [-1, -1, 1]
    assert f.replay is not None


def a_lists_values_are_no_key():
    """A contraction with a list of numbers is laid out for no one: the table neither grows with its values nor holds them."""
    t = f32([1, 2], [3, 4])
    Hip.dot, plain = classmethod(lambda cls, out, *args: out.with_(data=t.data)), Hip.dot.__func__
    for i in range(20):
        Nx.dot(t, [float(i), 1.0])
        Nx.dot(t, np.array([1.0, float(i)], np.float32))
        Nx.dot(t, [1], [float(i), 2.0], [0])
    assert len(Nx._ready) == 0, list(Nx._ready)
    for axes in ([1], (1,)):
        Nx.dot(t, axes, t, axes)
    assert len(Nx._ready) <= 1
    # the plans that a call is laid out from may be gone, cleared by another thread
    Hip.dot, Hip._dot_plans = classmethod(plain), {}
    assert Hip.prepared("dot", "dot", t.with_(data=None), t, [1], [], t, [1], []) is None


def a_refused_attempt_is_not_made_again():
    """What the library does not take at these extents is known from the first refusal on: no buffer is made for it again, and none
    is part of a recording."""
    q = from_numpy(np.ones((2, 4, 6, 8), np.float32), "f32", Hip)
    out = q.with_(data=None, shape=(2, 6, 4, 4))
    for _ in range(3):
        raises(lambda: Hip.dot_views(out, q, (0, 2, 1, 3), [3], [0, 1], q, (0, 2, 1, 3), [3], [0, 1]), "")
    assert standin.counts.get("hipnx_dot_strided") == 1
    b = from_numpy(np.ones((2, 4, 6, 64), np.uint16), "bf16", Hip)
    out = b.with_(data=None, type="f32", shape=(2, 6, 4, 4))
    program, layout = defn._Program([{"kind": B.L.FUSED_SET, "src": B.L.FUSED_SRC_INPUT, "dt": ("f", 32)}]), (48, 4, [(4, 1)])
    before = dict(standin.counts)
    for _ in range(3):
        raises(lambda: Hip.fused_scores(out, program, [b], layout, 0, (b, (0, 2, 1, 3), [3], [0, 1], b, (0, 2, 1, 3), [3], [0, 1]), mode="compiled"), "")
    assert standin.counts["hipnx_fused_scores"] == 1 and standin.counts["hipnx_buf_alloc"] == before["hipnx_buf_alloc"] + 1
    B._capturing.add(0)      # (a program is not compiled while capturing, whatever its extents)
    program = defn._Program(program)
    raises(lambda: Hip.fused_scores(out, program, [b], layout, 0, (b, (0, 2, 1, 3), [3], [0, 1], b, (0, 2, 1, 3), [3], [0, 1]), mode="compiled"), "")
    B._capturing.discard(0)
    raises(lambda: Hip.fused_scores(out, program, [b], layout, 0, (b, (0, 2, 1, 3), [3], [0, 1], b, (0, 2, 1, 3), [3], [0, 1]), mode="compiled"), "")
    assert standin.counts["hipnx_fused_scores"] == 3


def a_number_laid_out_with_its_call_is_that_number():
    """Numbers of both kinds, zeros of both signs, other tensors, other default backends, more numbers than are kept."""
    x, y = f32(1, 2, 4), f32(3, 5, 7)
    for _ in range(4):
        assert read(Nx.multiply(x, 0.5)) == [0.5, 1, 2] and read(Nx.multiply(y, 0.5)) == [1.5, 2.5, 3.5] and read(Nx.multiply(x, 3)) == [3, 6, 12]
        assert read(Nx.multiply(x, 3.0)) == [3, 6, 12] and str(read(Nx.multiply(x, 0.0))) == "[0.0, 0.0, 0.0]"
        assert str(read(Nx.multiply(x, -0.0))) == "[-0.0, -0.0, -0.0]" and read(Nx.multiply(x, True)) == [1, 2, 4]
        assert all(v != v for v in read(Nx.add(x, float("nan"))))
    assert any(k[1] == 0.5 for k in Nx._bound) and not any(k[1] == 0 for k in Nx._bound)
    gone = f32(1, 2, 4)
    assert Nx.backend_deallocate(gone) == "ok"
    raises(lambda: Nx.multiply(gone, 0.5), "deallocated")
    for i in range(3000):
        assert read(Nx.add(x, i + 0.5)) == [1 + i + 0.5, 2 + i + 0.5, 4 + i + 0.5]
    assert len(Nx._bound) <= 1024 and read(Nx.multiply(x, 0.5)) == [0.5, 1, 2]
    previous = B.bf16_rounding("nearest_even")
    assert not Nx._bound and read(Nx.multiply(x, 0.5)) == [0.5, 1, 2]
    B.bf16_rounding(previous)
    for _ in range(3):
        Nx.multiply(x, 0.5)
    Nx.default_backend(HostBinary)  # (its constants follow the tensor: no number of the device's is taken for one of its own)
    assert read(Nx.multiply(x, 0.5)) == [0.5, 1, 2]
    Nx.default_backend(Hip)


def a_number_is_laid_out_when_it_is_met_again():
    """Numbers that are met once are not laid out, whatever their number, and leave those that are alone; NaN never is; a call that a
    change of setting overtakes goes where nobody looks."""
    x = f32(1, 2, 4)
    for _ in range(4):
        assert read(Nx.multiply(x, 0.5)) == [0.5, 1, 2]
    assert [k[1] for k in Nx._bound] == [0.5]
    kept = Nx._bound[next(iter(Nx._bound))]
    for i in range(3000):
        assert read(Nx.multiply(x, i + 0.25)) == [i + 0.25, 2 * i + 0.5, 4 * i + 1]
        assert all(v != v for v in read(Nx.multiply(x, float("nan"))))
    nan = float("nan")
    for _ in range(4):
        assert all(v != v for v in read(Nx.multiply(x, nan)))
    assert list(Nx._bound.values()) == [kept] and len(Nx._met) <= 1024
    for i in range(1200):  # (each met again: the oldest go, not all of them)
        for _ in range(2):
            Nx.multiply(x, i + 0.125)
    assert 900 < len(Nx._bound) <= 1024 and any(k[1] == 1199.125 for k in Nx._bound)
    for name, value in list(Nx._ready.items()):
        if name[0] == "multiply":
            class Overtaken:
                def __call__(self, *args):
                    B._settings_changed()
                    return value(*args)

                def bind(self, *args):
                    return value.bind(*args)
            Nx.multiply(x, 9000.5)  # (met once)
            Nx._ready[name] = Overtaken()
            assert read(Nx.multiply(x, 9000.5)) == [9000.5, 18001, 36002]
            assert not Nx._bound and not Nx._ready
            break
    else:
        raise AssertionError("no product is laid out")


def what_a_recording_was_not_made_for_is_evaluated_or_refused():
    """Arguments of other types, shapes and kinds go the general way, with what it says of them."""
    x, y = f32(1, 2, 4), f32(3, 5, 7)
    f = defn.compile(lambda a, b: (Nx.add(a, b), Nx.multiply(a, 2.0)), x, y)
    for _ in range(5):
        total, twice = f(x, y)
    assert f.replay is not None and read(total) == [4, 7, 11] and read(twice) == [2, 4, 8]
    raises(lambda: f(x, f32(1, 2)), "traced for")
    raises(lambda: f(x, from_numpy(np.asarray([1, 2, 4], np.int32), "s32", Hip)), "traced for")
    raises(lambda: f(x), "expected 2")
    raises(lambda: f(x, y, y), "expected 2")
    one = defn.compile(lambda a, s: Nx.multiply(a, s), x, 2.0)
    for k in range(6):
        assert read(one(x, float(k))) == [k, 2 * k, 4 * k]
    pair = defn.compile(lambda ab: {"d": Nx.subtract(ab[0], ab[1])}, (x, y))
    for _ in range(6):
        assert read(pair((x, y))["d"]) == [-2, -3, -3]


def a_lender_that_holds_what_it_lent_to_is_collected():
    import gc
    import weakref

    class Lender:
        pass
    owner = f32(1, 2, 4)
    lender = Lender()
    lender.tensor = Nx.from_pointer(Hip, Nx.Pointer(kind="local", address=Nx.to_pointer(owner).address, data_size=12), "f32", (3,), keep=lender)
    assert read(lender.tensor) == [1, 2, 4]
    gone, handles = weakref.ref(lender), len(standin.memory)
    del lender
    gc.collect()
    assert gone() is None and len(standin.memory) == handles - 1
    assert read(owner) == [1, 2, 4]


if __name__ == "__main__":
    globals()[sys.argv[1]]()
