"""Traced functions evaluated on the device: the callers one step above the callbacks
(nx/lib/nx/defn/evaluator.ex:363-388).  The device runs the traced function, the oracle runs the
same function eagerly and traced; exact ops are compared bit for bit, transcendental chains within
the tolerances of the per-op tests."""
import gc

import numpy as np
import pytest

from nx_amd.tensor import template

from nx_amd import defn
from nx_amd import nx as Nx
from nx_amd import random as Random
from nx_amd import _lib as L
from nx_amd.backend import _Context, mem_stats
from random_support import CASES, check_random_case
from support import assert_all_close, assert_bits_equal, from_numpy, raw, seed_of
from test_defn import CHAINS, build_args, f32

pytestmark = pytest.mark.gpu

EXACT = {"linear_int8", "argmax_take"}  # integer dot, conversion, one float multiply; selection and copy


@pytest.mark.parametrize("name", sorted(CHAINS))
def test_jitted_chain_on_the_device(name, hip, oracle):
    got = defn.jit(CHAINS[name])(*build_args(hip)[name])
    assert type(got.data) is hip
    want = CHAINS[name](*build_args(oracle)[name])
    if name in EXACT:
        assert_bits_equal(got, want, name)
    else:
        assert_all_close(got, want, 1e-5, 1e-7, name)
    compiled = defn.compile(CHAINS[name], *build_args(hip)[name])
    again = compiled(*build_args(hip)[name])
    assert_bits_equal(again, got, f"{name}: compiled once, same result")


def test_constants_and_created_tensors_follow_the_arguments(hip):
    # the default backend only stores data here: iota and constants of the trace go to the device
    def fun(t):
        return Nx.add(Nx.multiply(t, Nx.iota((4,), type="f32")), 2.5)
    got = defn.jit(fun)(f32([1, 2, 3, 4], hip))
    assert type(got.data) is hip and hip.to_numpy(got).tolist() == [2.5, 4.5, 8.5, 14.5]


def test_control_flow_on_the_device(hip, oracle):
    def newton_sqrt(a):
        def body(state):
            i, x = state
            return Nx.add(i, 1), Nx.multiply(0.5, Nx.add(x, Nx.divide(a, x)))
        _, x = defn.while_loop((Nx.tensor(0), a), lambda s: Nx.less(s[0], 8), body)
        return defn.cond(Nx.greater(Nx.reduce_max(a), 100.0), lambda: Nx.negate(x), lambda: x)
    values = np.asarray([1.0, 2.0, 9.0, 50.0], dtype=np.float32)
    got = defn.jit(newton_sqrt)(f32(values, hip))
    want = defn.jit(newton_sqrt)(f32(values, oracle))
    assert_bits_equal(got, want, "newton sqrt")  # add, multiply, divide: exactly rounded
    flipped = defn.jit(newton_sqrt)(f32(values * 10, hip))
    assert (hip.to_numpy(flipped) < 0).all()


def test_intermediates_go_back_to_the_pool_during_the_walk(hip):
    n = 1 << 22  # 16 MiB per f32 intermediate
    x = from_numpy(np.linspace(0, 1, n, dtype=np.float32), "f32", hip)

    def chain(t):
        for _ in range(12):
            t = Nx.exp(Nx.negate(t))
        return t
    gc.collect()  # tensors earlier tests left behind must not be freed in the middle of the walk,
    L.check(L.lib.hipnx_trim(_Context.get(0)))  # nor their larger pooled blocks be handed out for these 16 MiB
    defn.jit(chain)(x)  # warm the pool
    before = mem_stats()["live"]
    seen = []
    original = defn._Run.apply

    def sampling(self, e, node, scope):
        seen.append(mem_stats()["live"] - before)
        return original(self, e, node, scope)
    defn._Run.apply = sampling
    try:
        out = defn.jit(chain)(x)
    finally:
        defn._Run.apply = original
    assert type(out.data) is hip
    # 24 intermediates of 16 MiB: with every result dropped after its last use at most the operand in
    # flight (and the result being written) is alive at any step, never the whole chain
    assert max(seen) <= 2 * 4 * n + 4096, seen
    assert mem_stats()["live"] - before <= 4 * n + 4096  # only the output stays


@pytest.mark.parametrize("case", [c for c in CASES if c["fn"] != "key"], ids=[c["name"] for c in CASES if c["fn"] != "key"])
def test_random_known_answers_through_a_trace_on_the_device(case, hip):
    check_random_case(case, hip, through=defn.jit)


def test_traced_random_uses_the_one_kernel_cipher(hip):
    key = Random.key(99, backend=hip)
    traced = defn.jit(lambda k: Random.random_bits(k, shape=(1001,)))(key)
    previous = Random.compose_only(True)
    try:
        composed = Random.random_bits(key, shape=(1001,))
    finally:
        Random.compose_only(previous)
    assert_bits_equal(traced, composed, "random_bits traced vs composed")


# ---- captured graphs: one submission replays every kernel of a compiled function ------------------

# (argmax_take too: indices written by argmax are known to be in range of an axis of that length, so take's raising
# bounds policy has nothing to wait for)
GRAPHABLE = ["softmax", "elementwise_reduce", "linear_int8", "argmax_take"]


@pytest.mark.parametrize("name", GRAPHABLE)
def test_captured_chain_replays_with_new_inputs(name, hip):
    from nx_amd.backend import sync
    args = build_args(hip)[name]
    compiled = defn.compile(CHAINS[name], *args)
    eager = hip.to_numpy(compiled(*args)).copy()
    captured = compiled.capture(*args)
    try:
        # replays between eager work and synchronisations, every one checked against the eager result
        for _ in range(3):
            out = captured(*args)
            np.testing.assert_array_equal(hip.to_numpy(out), eager, f"{name}: replay with the captured tensors")
            compiled(*args)
            sync()
        # new values in fresh tensors of the same shapes: copied in, same kernels
        rng = np.random.default_rng(11)
        fresh = []
        for a in args:
            raw = hip.to_numpy(a)
            perm = rng.permutation(raw.size)
            fresh.append(from_numpy(raw.reshape(-1)[perm].reshape(raw.shape), a.type, hip))
        want = hip.to_numpy(compiled(*fresh)).copy()
        np.testing.assert_array_equal(hip.to_numpy(captured(*fresh)), want, f"{name}: replay with new inputs")
        np.testing.assert_array_equal(hip.to_numpy(captured(*args)), eager, f"{name}: and back")
    finally:
        captured.destroy()


def test_captured_constants_survive_the_scalar_cache(hip):
    """A constant met while capturing is the graph's own block, filled inside the capture -- also when the
    eager warm-up has left the same number in the backend's scalar cache.  After more than 1024 other
    scalars have passed through that cache (it is cleared, its blocks go back to the pool and are
    overwritten), a replay still multiplies by 0.5."""
    x_np = np.linspace(-3, 3, 4096, dtype=np.float32)
    x = from_numpy(x_np, "f32", hip)
    compiled = defn.compile(lambda t: Nx.add(Nx.multiply(t, 0.5), 0.25), x)
    want = hip.to_numpy(compiled(x)).copy()  # the warm-up: 0.5 and 0.25 are now cached scalars
    captured = compiled.capture(x)
    try:
        np.testing.assert_array_equal(hip.to_numpy(captured(x)), want)
        keep = []
        for i in range(1100):  # distinct scalars: the cache overflows and is cleared
            keep.append(Nx.multiply(x, 1.0 + i / 4096.0))
        del keep
        junk = [hip.constant(template("f32", ()), 1000.0 + i, {}) for i in range(64)]  # take the freed small blocks
        np.testing.assert_array_equal(hip.to_numpy(captured(x)), want, "replay after the cache was cleared")
        del junk
    finally:
        captured.destroy()


def test_capture_refuses_what_needs_the_host(hip):
    """`take` with indices from outside (an argument: nothing is known about them) under the raising bounds policy has
    to wait for its kernel, which a capture cannot."""
    from nx_amd._lib import HipNxError
    rng = np.random.default_rng(3)
    table = from_numpy((rng.standard_normal((100, 24)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16), "bf16", hip)
    idx = from_numpy(rng.integers(0, 100, size=16, dtype=np.uint32), "u32", hip)
    compiled = defn.compile(lambda t, i: Nx.take(t, i), table, idx)
    with pytest.raises(HipNxError, match="not possible while capturing"):
        compiled.capture(table, idx)
    # the failed capture leaves the context usable
    assert_bits_equal(compiled(table, idx), Nx.take(table, idx), "eager after a refused capture")


def test_graph_blocks_do_not_leak_into_the_pool(hip):
    n = 1 << 20
    x = from_numpy(np.linspace(-1, 1, n, dtype=np.float32), "f32", hip)

    def chain(t):
        for _ in range(6):
            t = Nx.exp(Nx.negate(t))
        return t
    compiled = defn.compile(chain, x)
    want = hip.to_numpy(compiled(x)).copy()
    captured = compiled.capture(x)
    out = captured(x)
    # eager work of the same sizes in between must not be handed the graph's blocks
    others = [Nx.exp(x) for _ in range(8)]
    np.testing.assert_array_equal(hip.to_numpy(captured(x)), want)
    np.testing.assert_array_equal(hip.to_numpy(others[0]), hip.to_numpy(Nx.exp(x)))
    del others, out
    before = mem_stats()
    captured.destroy()
    after = mem_stats()
    assert after["pooled"] >= before["pooled"]  # the graph's blocks return to the pool only now
    np.testing.assert_array_equal(hip.to_numpy(compiled(x)), want)


# ---- fused element-wise groups: one kernel per group, the same bits as node by node -----------------

def gelu_like(x, bias):
    h = Nx.add(x, bias)
    return Nx.multiply(Nx.multiply(h, 0.5), Nx.add(1.0, Nx.tanh(Nx.multiply(0.7978845608, Nx.add(h, Nx.multiply(0.044715, Nx.pow(h, 3.0)))))))


def relu_mask(x, y):
    keep = Nx.logical_and(Nx.greater(x, 0.0), Nx.less_equal(y, 0.5))
    return Nx.select(keep, Nx.sqrt(Nx.abs(x)), Nx.negate(y))


def mixed_precision(a, b):
    # every intermediate rounds to its own type: bf16 by truncation, f16 to nearest
    h = Nx.multiply(a, b)                       # bf16 * f16 -> f16? no: merged float type
    return Nx.as_type(Nx.exp(Nx.as_type(Nx.add(h, 0.25), "bf16")), "f16")


def row_and_column_operands(x, row, col):
    return Nx.divide(Nx.subtract(x, col), Nx.add(row, 1.5))


def rand_float(rng, ty, shape, backend):
    v = rng.standard_normal(shape).astype(np.float32)
    if ty == "bf16":
        return from_numpy((v.view(np.uint32) >> 16).astype(np.uint16), "bf16", backend)
    return from_numpy(v.astype(np.float16 if ty == "f16" else np.float32), ty, backend)


def reuse_and_square(x, y):
    s = Nx.add(x, y)
    return Nx.multiply(Nx.multiply(s, s), Nx.subtract(s, x))   # op(s, s) and three reads of one value


def masked_products(x, y):
    kept = Nx.greater(x, 0.0)
    return Nx.subtract(Nx.multiply(kept, Nx.add(x, y)), Nx.multiply(Nx.multiply(y, Nx.is_nan(Nx.divide(x, x))), kept))


def product_with_a_given_mask(x, y, mask):
    return Nx.multiply(Nx.add(x, y), mask)


def not_finite(rng, ty, shape, b):
    v = rng.standard_normal(shape).astype(np.float32)
    v.reshape(-1)[::3] = np.resize(np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40], np.float32), v.reshape(-1)[::3].shape)
    return from_numpy((v.view(np.uint32) >> 16).astype(np.uint16) if ty == "bf16" else v.astype(np.float16 if ty == "f16" else np.float32), ty, b)


FUSED_CASES = {
    "masked_products": (masked_products, lambda rng, b: (not_finite(rng, "f32", (64, 40), b), not_finite(rng, "f32", (64, 40), b))),
    "masked_products_ragged": (masked_products, lambda rng, b: (not_finite(rng, "f16", (13, 7), b), not_finite(rng, "f16", (13, 7), b))),
    "product_with_a_given_mask": (product_with_a_given_mask, lambda rng, b: (not_finite(rng, "bf16", (24, 64), b), not_finite(rng, "bf16", (24, 64), b),
                                                                             from_numpy(rng.integers(0, 256, size=(24, 64), dtype=np.uint8), "u8", b))),
    "reuse_and_square": (reuse_and_square, lambda rng, b: (rand_float(rng, "f32", (40, 64), b), rand_float(rng, "f32", (40, 64), b))),
    "long_rows_tail": (gelu_like, lambda rng, b: (rand_float(rng, "f32", (3, 4104), b), rand_float(rng, "f32", (4104,), b))),
    "gelu_like": (gelu_like, lambda rng, b: (rand_float(rng, "f32", (64, 256), b), rand_float(rng, "f32", (256,), b))),
    "gelu_like_bf16": (gelu_like, lambda rng, b: (rand_float(rng, "bf16", (8, 16, 128), b), rand_float(rng, "bf16", (128,), b))),
    "relu_mask": (relu_mask, lambda rng, b: (rand_float(rng, "f32", (1000, 24), b), rand_float(rng, "f32", (1000, 24), b))),
    "relu_mask_ragged": (relu_mask, lambda rng, b: (rand_float(rng, "f32", (37, 11), b), rand_float(rng, "f32", (37, 11), b))),
    "mixed_precision": (mixed_precision, lambda rng, b: (rand_float(rng, "bf16", (33, 40), b), rand_float(rng, "f16", (33, 40), b))),
    "row_and_column": (row_and_column_operands, lambda rng, b: (rand_float(rng, "f32", (48, 64), b), rand_float(rng, "f32", (64,), b),
                                                                 rand_float(rng, "f32", (48, 1), b))),
    "row_and_column_unaligned": (row_and_column_operands, lambda rng, b: (rand_float(rng, "f32", (5, 7), b), rand_float(rng, "f32", (7,), b),
                                                                           rand_float(rng, "f32", (5, 1), b))),
}


@pytest.fixture(params=["interpreted", "compiled"])
def fused_mode(request, hip):
    """Runs a test once with the interpreting kernels and once with each program compiled at run time."""
    from nx_amd.backend import fused_mode as set_mode
    set_mode(request.param)
    yield request.param
    set_mode("interpreted")


@pytest.mark.parametrize("name", sorted(FUSED_CASES))
def test_fused_group_is_bit_identical_to_node_by_node(name, hip, fused_mode):
    fun, make = FUSED_CASES[name]
    args = make(np.random.default_rng(3), hip)
    fused = defn.compile(fun, *args, fuse=True)
    assert fused.fused_groups >= 1
    assert_bits_equal(fused(*args), defn.compile(fun, *args)(*args), name)


@pytest.mark.parametrize("name", sorted(CHAINS))
def test_fused_configuration_chains(name, hip, fused_mode):
    args = build_args(hip)[name]
    assert_bits_equal(defn.compile(CHAINS[name], *args, fuse=True)(*args), defn.compile(CHAINS[name], *args)(*args), name)


def test_fused_kernel_is_the_path_taken(hip):
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        calls.append(1)
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        fun, make = FUSED_CASES["gelu_like"]
        args = make(np.random.default_rng(5), hip)
        defn.compile(fun, *args, fuse=True)(*args)
    finally:
        hip.fused_elementwise = classmethod(original)
    assert calls == [1]  # the whole function is one group


def test_fused_entry_point_validates_its_program(hip):
    from nx_amd._lib import FUSED_BINARY, FUSED_SET, FUSED_SRC_INPUT, FUSED_SRC_SAVED, FUSED_UNARY, HipNxError
    x = rand_float(np.random.default_rng(1), "f32", (16,), hip)
    out = x.with_(data=None)
    flat = (1, 16, [(0, 1)])
    load = {"kind": FUSED_SET, "src": FUSED_SRC_INPUT, "arg": 0, "dt": ("f", 32)}
    with pytest.raises(HipNxError, match="before anything set it"):
        hip.fused_elementwise(out, [{"kind": FUSED_UNARY, "op": 0, "dt": ("f", 32)}], [x], flat)
    with pytest.raises(HipNxError, match="reads an input that is not there"):
        hip.fused_elementwise(out, [dict(load, arg=3)], [x], flat)
    with pytest.raises(HipNxError, match="reads an empty slot"):
        hip.fused_elementwise(out, [load, {"kind": FUSED_BINARY, "op": 0, "src": FUSED_SRC_SAVED, "arg": 1, "dt": ("f", 32)}], [x], flat)
    with pytest.raises(HipNxError, match="binary op"):
        hip.fused_elementwise(out, [load, {"kind": FUSED_BINARY, "op": 9, "src": FUSED_SRC_INPUT, "arg": 0, "dt": ("f", 32)}], [x], flat)
    with pytest.raises(HipNxError, match="holds"):
        hip.fused_elementwise(out.with_(shape=(32,)), [load], [x], (1, 32, [(0, 1)]))
    got = hip.fused_elementwise(out, [load, {"kind": FUSED_UNARY, "op": 27, "dt": ("f", 32)}], [x], flat)  # negate
    np.testing.assert_array_equal(hip.to_numpy(got), -hip.to_numpy(x))


def test_each_distinct_program_is_compiled_once(hip):
    from nx_amd.backend import fused_compiled_count, fused_mode as set_mode
    fun, make = FUSED_CASES["relu_mask"]
    args = make(np.random.default_rng(8), hip)
    other = tuple(rand_float(np.random.default_rng(9), "f32", (16, 128), hip) for _ in range(2))
    want = defn.compile(fun, *args)(*args)
    set_mode("compiled")
    try:
        before = fused_compiled_count()
        fused = defn.compile(fun, *args, fuse=True)
        assert_bits_equal(fused(*args), want, "first call compiles")
        after = fused_compiled_count()
        assert after >= before  # `before + 1` unless an earlier test met the same program
        assert_bits_equal(fused(*args), want, "second call reuses")
        defn.compile(fun, *other, fuse=True)(*other)  # other shape, same program: the shape is not compiled in
        assert fused_compiled_count() == after
        set_mode("interpreted")
        assert_bits_equal(fused(*args), want, "and back")
    finally:
        set_mode("interpreted")


def test_compiled_programs_are_bounded_and_the_oldest_go_first(hip):
    """A constant is part of what a program is compiled for, so a number that changes per call makes a new
    program each time: the table stops at its limit, and a program unloaded meanwhile compiles again."""
    from nx_amd import backend as B
    from nx_amd._lib import HipNxError
    x = rand_float(np.random.default_rng(12), "f32", (32, 64), hip)
    xs = hip.to_numpy(x)

    def scaled(c):
        def fun(t):
            return Nx.multiply(Nx.tanh(t), c)
        return fun
    consts = [1.0 + i / 16 for i in range(1, 11)]  # (not 1.0: the tracer drops a multiplication by one, and the first call must compile)
    B.fused_mode("compiled")
    B.fused_cache_limit(8)
    pinned = 4  # programs that earlier tests recorded into graphs stay loaded
    try:
        for c in consts + consts[:2]:  # the first two have been unloaded by the time they come round again
            got = hip.to_numpy(defn.compile(scaled(c), x, fuse=True)(x))
            want = (np.tanh(xs.astype(np.float64)).astype(np.float32) * np.float32(c))
            np.testing.assert_allclose(got, want, rtol=2e-6)
            assert B.fused_compiled_count() <= 8 + pinned
        with pytest.raises(HipNxError, match="at least 4"):
            B.fused_cache_limit(1)
    finally:
        B.fused_cache_limit(512)
        B.fused_mode("interpreted")


def test_program_first_met_during_a_capture_runs_interpreted(hip):
    from nx_amd import backend as B

    def fresh(x, y):  # a program no other test builds
        return Nx.subtract(Nx.multiply(Nx.sigmoid(x), 1.25), Nx.floor(y))
    args = tuple(rand_float(np.random.default_rng(10), "f32", (64, 64), hip) for _ in range(2))
    want = defn.compile(fresh, *args)(*args)
    fused = defn.compile(fresh, *args, fuse=True)
    fused(*args)  # the run before a capture, as the capture rules ask -- interpreted, so nothing is compiled yet
    B.fused_mode("compiled")
    try:
        before = B.fused_compiled_count()
        B.capture_begin(0)
        try:
            out = fused(*args)
        finally:
            graph = B.capture_end(0)
        assert B.fused_compiled_count() == before  # compiling and loading a module is no work to record
        for _ in range(3):
            graph.launch()
            assert_bits_equal(out, want, "replay")
        del out
        graph.destroy()
        assert_bits_equal(fused(*args), want, "compiled after the capture")
        assert B.fused_compiled_count() == before + 1
    finally:
        B.fused_mode("interpreted")


# ---- a reduction over the last axis joins the group that feeds it ----------------------------------------

def sum_of_exp(a, b):
    return Nx.sum(Nx.exp(Nx.multiply(Nx.add(a, b), 0.5)), axes=[1])


def max_of_scaled(a, b):
    return Nx.reduce_max(Nx.multiply(Nx.subtract(a, b), 0.125), axes=[-1], keep_axes=True)


def min_of_bf16(a, b):
    return Nx.reduce_min(Nx.as_type(Nx.add(a, b), "bf16"), axes=[1])


def sum_of_sines(a, b):  # sin is outside the light instantiation of the interpreting kernels
    return Nx.sum(Nx.sin(Nx.add(a, b)), axes=[1])


REDUCED = {"sum_of_exp": sum_of_exp, "max_of_scaled": max_of_scaled, "min_of_bf16": min_of_bf16}


def test_compiled_reduction_takes_any_float_program(hip):
    from nx_amd.backend import fused_mode as set_mode
    rng = np.random.default_rng(21)
    args = (rand_float(rng, "f32", (96, 512), hip), rand_float(rng, "f32", (96, 512), hip))
    want = defn.compile(sum_of_sines, *args)(*args)
    fused = defn.compile(sum_of_sines, *args, fuse=True)
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        calls.append(a[4] if len(a) > 4 else k.get("reduce_op", -1))
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        assert_bits_equal(fused(*args), want, "interpreted: the group, then the separate reduction")
        assert calls == [0, -1]  # offered with the reduction, refused, run without it
        del calls[:]
        set_mode("compiled")
        assert_bits_equal(fused(*args), want, "compiled: one kernel")
        assert calls == [0]
    finally:
        set_mode("interpreted")
        hip.fused_elementwise = classmethod(original)


@pytest.mark.parametrize("name", sorted(REDUCED))
@pytest.mark.parametrize("shape", [(64, 256), (300, 4096), (16, 8192), (5, 40000), (4, 65536), (1, 1000000), (2, 131080), (2049, 8),
                                   (3, 7, 512)])
def test_group_with_its_row_reduction_is_bit_identical(name, shape, hip, fused_mode):
    rng = np.random.default_rng(seed_of(name, shape))
    if len(shape) == 3 and name == "sum_of_exp":
        pytest.skip("this function reduces axis 1, which is the last axis only for matrices")
    fun = REDUCED[name]
    if len(shape) == 3 and name == "min_of_bf16":
        fun = lambda a, b: Nx.reduce_min(Nx.as_type(Nx.add(a, b), "bf16"), axes=[2])  # noqa: E731
    args = (rand_float(rng, "f32", shape, hip), rand_float(rng, "f32", shape, hip))
    fused = defn.compile(fun, *args, fuse=True)
    assert fused.fused_groups == 1 and fused.roots[0].data.op == "fused" and fused.roots[0].data.args[0].reduce is not None
    assert_bits_equal(fused(*args), defn.compile(fun, *args)(*args), f"{name} {shape}")


def fused_groups_of(compiled):
    groups = []

    def seen(t):
        e = t.data
        if e.op == "fused":
            groups.append(e.args[0])
            for i in e.args[1]:
                seen(i)
        elif e.op not in ("parameter", "constant", "tensor"):
            for ch in defn._children(e):
                if isinstance(ch, defn.Tensor):
                    seen(ch)
    for r in compiled.roots:
        seen(r)
    return groups


def test_softmax_becomes_three_kernels(hip, fused_mode):
    """The scaled scores feed the max and the subtraction, the exponentials feed the sum and the
    division: both are cheap to compute again from the bf16 scores, so nothing but the two row
    statistics and the result is ever stored."""
    args = build_args(hip)["softmax"]
    fused = defn.compile(CHAINS["softmax"], *args, fuse=True)
    assert_bits_equal(fused(*args), defn.compile(CHAINS["softmax"], *args)(*args), "softmax")
    groups = fused_groups_of(fused)
    assert sorted(str(g.reduce and g.reduce[0]) for g in {id(g): g for g in groups}.values()) == ["None", "reduce_max", "sum"]
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        calls.append(1)
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        fused(*args)
    finally:
        hip.fused_elementwise = classmethod(original)
    assert len(calls) == 3


def test_value_with_an_outside_reader_is_still_stored_once(hip):
    x = rand_float(np.random.default_rng(2), "f32", (32, 64), hip)

    def fun(t):
        h = Nx.tanh(Nx.multiply(t, 0.5))
        return Nx.add(h, 1.0), Nx.dot(h, [1], h, [1])   # the dot is not element-wise: h must exist in memory
    fused = defn.compile(fun, x, fuse=True)
    plain = defn.compile(fun, x)
    for got, want in zip(fused(x), plain(x)):
        assert_bits_equal(got, want, "shared with a dot")


# ---- groups planned for compilation: 32-bit integer work and bit relabelling join in --------------------

def bits_to_unit_floats(bits):
    # the core of Nx.Random.uniform for f32 (random.ex:424-470): mantissa bits under the exponent of 1.0
    mantissa = Nx.bitwise_or(Nx.right_shift(bits, 9), 0x3F800000)
    return Nx.subtract(Nx.bitcast(mantissa, "f32"), 1.0)


def integer_mix(a, b):
    x = Nx.bitwise_xor(Nx.add(a, b), Nx.left_shift(a, 3))
    return Nx.multiply(Nx.subtract(x, 7), Nx.bitwise_not(b))


def signed_shift_and_convert(a, b):
    x = Nx.max(Nx.right_shift(Nx.negate(a), 2), Nx.min(b, 1000))
    return Nx.multiply(Nx.as_type(x, "f32"), 0.5)


def floats_to_bits_and_back(x):
    sign_cleared = Nx.bitwise_and(Nx.bitcast(x, "u32"), 0x7FFFFFFF)
    return Nx.sqrt(Nx.bitcast(sign_cleared, "f32"))


# Where the bits of a float can be looked at, every NaN a node computes is the one quiet NaN its kernel would have stored
# (0x7FC00000), bits that only pass through a relabelling stay as they are, and a conversion rounds however few significant
# bits the compiler can see in the integer (each of these once came out differently from the compiled group):
def bits_of_a_computed_nan(x):
    return Nx.bitcast(Nx.sqrt(x), "s32")                       # sqrt of a negative number: the hardware's NaN has the sign set


def relabelled_nan_bits(a):
    return Nx.bitcast(Nx.negate(Nx.max(a, 0x7FFFFFFF)), "f32")  # NaN patterns with payloads: the result's last node relabels


def shifted_integer_to_f16(a):
    return Nx.sqrt(Nx.as_type(Nx.left_shift(a, 24), "f16"))     # eight significant bits, far beyond f16's range: infinity


def sign_extended_byte_as_float(a):
    return Nx.subtract(Nx.bitcast(Nx.right_shift(a, 24), "f32"), 1.0)   # negative a: the bits of a NaN


def rand_words(rng, ty, shape, backend):
    info = np.iinfo(np.uint32 if ty == "u32" else np.int32)
    return from_numpy(rng.integers(info.min, info.max, size=shape, dtype=info.dtype, endpoint=True), ty, backend)


INT_CASES = {
    "bits_to_unit_floats": (bits_to_unit_floats, lambda rng, b: (rand_words(rng, "u32", (64, 256), b),)),
    "integer_mix_u32": (integer_mix, lambda rng, b: (rand_words(rng, "u32", (33, 128), b), rand_words(rng, "u32", (33, 128), b))),
    "integer_mix_s32": (integer_mix, lambda rng, b: (rand_words(rng, "s32", (8, 4096), b), rand_words(rng, "s32", (4096,), b))),
    "signed_shift_and_convert": (signed_shift_and_convert, lambda rng, b: (rand_words(rng, "s32", (40, 64), b), rand_words(rng, "s32", (40, 64), b))),
    "floats_to_bits_and_back": (floats_to_bits_and_back, lambda rng, b: (rand_float(rng, "f32", (1000, 8), b),)),
    "bits_of_a_computed_nan": (bits_of_a_computed_nan, lambda rng, b: (rand_float(rng, "f32", (4, 64), b),)),
    "relabelled_nan_bits": (relabelled_nan_bits, lambda rng, b: (rand_words(rng, "u32", (5, 8), b),)),
    "shifted_integer_to_f16": (shifted_integer_to_f16, lambda rng, b: (rand_words(rng, "u32", (2, 520), b),)),
    "sign_extended_byte_as_float": (sign_extended_byte_as_float, lambda rng, b: (rand_words(rng, "s32", (64, 8), b),)),
}


def test_what_a_compiled_group_sees_in_the_bits_of_a_nan(hip):
    """The same four against what they must give, worked out here."""
    x = from_numpy(np.array([-4.0, 4.0, -0.0, -1e-30] * 2, np.float32), "f32", hip)
    got = raw(defn.compile(bits_of_a_computed_nan, x, fuse="compiled")(x))
    assert got.view(np.uint32).tolist() == [0x7FC00000, 0x40000000, 0x80000000, 0x7FC00000] * 2
    a = from_numpy(np.array([0x80000001, 0x7FFFFFFF, 5, 0xFFFFFFFF, 0x80000000, 0x80000002, 0, 9], np.uint32), "u32", hip)
    got = raw(defn.compile(relabelled_nan_bits, a, fuse="compiled")(a))
    assert got.view(np.uint32).tolist() == [0x7FFFFFFF, 0x80000001, 0x80000001, 1, 0x80000000, 0x7FFFFFFE, 0x80000001, 0x80000001]
    a = from_numpy(np.array([0, 1, 2, 255, 256 + 4, 16, 64, 100], np.uint32), "u32", hip)
    got = raw(defn.compile(shifted_integer_to_f16, a, fuse="compiled")(a))
    assert got.view(np.uint16).tolist() == [0, 0x7C00, 0x7C00, 0x7C00, 0x7C00, 0x7C00, 0x7C00, 0x7C00]
    a = from_numpy(np.array([-1 << 24, 3 << 24, -128 << 24, 0, 127 << 24, -5 << 24, 1 << 23, -(1 << 23)], np.int32), "s32", hip)
    got = raw(defn.compile(sign_extended_byte_as_float, a, fuse="compiled")(a))
    assert got.view(np.uint32).tolist() == [0x7FC00000, 0xBF800000, 0x7FC00000, 0xBF800000, 0xBF800000, 0x7FC00000, 0xBF800000, 0x7FC00000]


@pytest.mark.parametrize("name", sorted(INT_CASES))
def test_compiled_group_with_integer_work_is_bit_identical(name, hip):
    from nx_amd.backend import fused_mode as set_mode
    fun, make = INT_CASES[name]
    args = make(np.random.default_rng(seed_of(name)), hip)
    want = defn.compile(fun, *args)(*args)
    fused = defn.compile(fun, *args, fuse="compiled")
    assert fused.fused_groups == 1 and fused.roots[0].data.op == "fused"  # the whole function is one kernel
    assert_bits_equal(fused(*args), want, name)
    # planned without the integer class, the same function still agrees (float parts fuse, the rest runs node by node)
    assert_bits_equal(defn.compile(fun, *args, fuse=True)(*args), want, name + " float-only plan")
    set_mode("compiled")
    try:
        assert_bits_equal(fused(*args), want, name + " in compiled mode")
    finally:
        set_mode("interpreted")


def test_integer_program_is_refused_by_the_interpreting_kernels(hip):
    from nx_amd._lib import FUSED_BINARY, FUSED_SET, FUSED_SRC_CONST, FUSED_SRC_INPUT, HipNxError
    x = rand_words(np.random.default_rng(4), "u32", (64,), hip)
    program = [{"kind": FUSED_SET, "src": FUSED_SRC_INPUT, "arg": 0, "flags": 2, "dt": ("u", 32)},
               {"kind": FUSED_BINARY, "op": 14, "src": FUSED_SRC_CONST, "imm_bits": 9, "flags": 2, "dt": ("u", 32)}]  # right_shift
    with pytest.raises(HipNxError, match="need the compiled mode"):
        hip.fused_elementwise(x.with_(data=None), program, [x], (1, 64, [(0, 1)]))
    got = hip.fused_elementwise(x.with_(data=None), program, [x], (1, 64, [(0, 1)]), mode="compiled")
    np.testing.assert_array_equal(hip.to_numpy(got), hip.to_numpy(x) >> 9)


@pytest.mark.parametrize("name", ["uniform", "normal"])
def test_random_floats_from_one_compiled_group(name, hip):
    from nx_amd import random as Random
    key = Random.key(99, backend=hip)
    fun = {"uniform": lambda k: Random.uniform_split(k, -2.0, 3.0, shape=(64, 1024)),
           "normal": lambda k: Random.normal_split(k, 1.0, 2.0, shape=(64, 1024))}[name]
    want = defn.compile(fun, key)(key)
    fused = defn.compile(fun, key, fuse="compiled")
    assert_bits_equal(fused(key), want, name)
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        calls.append(1)
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        fused(key)
    finally:
        hip.fused_elementwise = classmethod(original)
    assert len(calls) >= 1 and fused.fused_groups == 1  # everything after the cipher is one group


# ---- dot -> as_type -> multiply by the scales on the accumulators (the quantised linear layer) -----------

def linear_scaled(xq, wq, sc):
    return Nx.multiply(Nx.as_type(Nx.dot(xq, [1], wq, [1], out_type="s32"), "f32"), sc)


def rand_s8(rng, shape, backend):
    return from_numpy(rng.integers(-127, 128, size=shape, dtype=np.int8), "s8", backend)


@pytest.mark.parametrize("m,n,k", [(64, 11008, 4096), (64, 256, 4096), (16, 512, 8192), (300, 520, 256), (256, 256, 128), (1024, 1024, 1024), (8, 40, 128)])
@pytest.mark.parametrize("scales", ["per_column", "per_row", "one", "constant"])
def test_scaled_int8_dot_is_bit_identical_to_the_three_callbacks(m, n, k, scales, hip):
    rng = np.random.default_rng(seed_of(m, n, k, scales))
    x, w = rand_s8(rng, (m, k), hip), rand_s8(rng, (n, k), hip)
    if scales == "constant":
        fun, args = (lambda xq, wq: linear_scaled(xq, wq, 0.0078125)), (x, w)
    else:
        shape = {"per_column": (n,), "per_row": (m, 1), "one": (1, 1)}[scales]
        sc = from_numpy(rng.uniform(1e-3, 1e-2, size=shape).astype(np.float32), "f32", hip)
        if scales == "per_column":  # a NaN and an infinity among the scales travel like in the multiply kernel
            raw = hip.to_numpy(sc).copy()
            raw[0], raw[-1] = np.nan, np.inf
            sc = from_numpy(raw, "f32", hip)
        fun, args = linear_scaled, (x, w, sc)
    want = defn.compile(fun, *args)(*args)
    planned = defn.compile(fun, *args, fuse=True)
    assert planned.roots[0].data.op == "dot_scaled"
    calls = []
    original = hip.dot_scaled.__func__

    def counting(cls, *a, **kw):
        calls.append(1)
        return original(cls, *a, **kw)
    hip.dot_scaled = classmethod(counting)
    try:
        assert_bits_equal(planned(*args), want, f"{m}x{n}x{k} {scales}")
    finally:
        hip.dot_scaled = classmethod(original)
    assert calls == [1]


def test_scaled_dot_with_batches_and_with_the_weights_k_outer(hip):
    rng = np.random.default_rng(77)
    x, w = rand_s8(rng, (4, 48, 256), hip), rand_s8(rng, (4, 256, 80), hip)
    sc = from_numpy(rng.uniform(1e-3, 1e-2, size=(80,)).astype(np.float32), "f32", hip)

    def fun(xq, wq, s):  # batched, the right operand contracted on its middle axis
        return Nx.multiply(Nx.as_type(Nx.dot(xq, [2], [0], wq, [1], [0], out_type="s32"), "f32"), s)
    planned = defn.compile(fun, x, w, sc, fuse=True)
    assert planned.roots[0].data.op == "dot_scaled"
    assert_bits_equal(planned(x, w, sc), defn.compile(fun, x, w, sc)(x, w, sc), "batched")


# partial slabs in place, rows copied to whole pieces, transposed first, both; fewer than 16 M multiply-adds: three calls
@pytest.mark.parametrize("M,N,K,contract", [(64, 512, 607, 1), (8, 4098, 607, 0), (33, 2000, 272, 0), (512, 300, 1008, 1), (128, 1040, 129, 0), (64, 640, 494, 1), (16, 32, 100, 1)])
@pytest.mark.parametrize("scales", ["column", "row", "one"])
def test_scaled_dot_of_any_k(M, N, K, contract, scales, hip):
    rng = np.random.default_rng(seed_of(M, N, K, contract, scales))
    x, w = rand_s8(rng, (M, K), hip), rand_s8(rng, (N, K) if contract else (K, N), hip)
    sc = from_numpy(rng.uniform(1e-3, 1e-2, size={"column": (N,), "row": (M, 1), "one": (1,)}[scales]).astype(np.float32), "f32", hip)

    def fun(xq, wq, s):
        return Nx.multiply(Nx.as_type(Nx.dot(xq, [1], wq, [contract], out_type="s32"), "f32"), s)
    planned = defn.compile(fun, x, w, sc, fuse="compiled")
    assert planned.roots[0].data.op == "dot_scaled"
    calls = []
    original = hip.as_type.__func__
    hip.as_type = classmethod(lambda cls, *a: (calls.append(1), original(cls, *a))[1])
    try:
        got = planned(x, w, sc)
    finally:
        hip.as_type = classmethod(original)
    assert bool(calls) == (M * N * K < 1 << 24 and (K % 16 != 0)), calls
    assert_bits_equal(got, defn.compile(fun, x, w, sc)(x, w, sc), f"{M} x {N} x {K}")


def test_scaled_dot_entry_point_refuses_what_it_does_not_take(hip):
    from nx_amd._lib import EUNSUPPORTED, SCALE_PER_COLUMN, HipNxError
    rng = np.random.default_rng(5)
    x, w = rand_s8(rng, (8, 100), hip), rand_s8(rng, (40, 100), hip)  # K is not a multiple of 128
    sc = from_numpy(np.ones(40, dtype=np.float32), "f32", hip)
    out = sc.with_(data=None, shape=(8, 40))
    with pytest.raises(HipNxError) as err:
        hip.dot_scaled(out, x, [1], [], w, [1], [], sc, SCALE_PER_COLUMN)
    assert err.value.status == EUNSUPPORTED
    # through the evaluator the same shapes make the three calls instead
    planned = defn.compile(linear_scaled, x, w, sc, fuse=True)
    assert_bits_equal(planned(x, w, sc), defn.compile(linear_scaled, x, w, sc)(x, w, sc), "fallback")
    short = from_numpy(np.ones(8, dtype=np.float32), "f32", hip)
    x2, w2 = rand_s8(rng, (16, 128), hip), rand_s8(rng, (40, 128), hip)
    with pytest.raises(HipNxError, match="holds"):
        hip.dot_scaled(sc.with_(data=None, shape=(16, 40)), x2, [1], [], w2, [1], [], short, SCALE_PER_COLUMN)


@pytest.mark.parametrize("K,contract", [(1000, 1), (1008, 1), (1009, 0)])
def test_scaled_dot_refuses_every_partial_slab_of_k(hip, K, contract):
    """Also where the plain contraction walks the partial slab in place or copies the rows: the three calls, same bits."""
    from nx_amd._lib import EUNSUPPORTED, SCALE_PER_COLUMN, HipNxError
    rng = np.random.default_rng(K)
    x, w = rand_s8(rng, (128, K), hip), rand_s8(rng, (144, K) if contract else (K, 144), hip)
    sc = from_numpy(rng.uniform(1e-3, 1e-2, size=(144,)).astype(np.float32), "f32", hip)
    with pytest.raises(HipNxError) as err:
        hip.dot_scaled(sc.with_(data=None, shape=(128, 144)), x, [1], [], w, [contract], [], sc, SCALE_PER_COLUMN)
    assert err.value.status == EUNSUPPORTED

    def fun(xq, wq, s):
        return Nx.multiply(Nx.as_type(Nx.dot(xq, [1], wq, [contract], out_type="s32"), "f32"), s)
    assert_bits_equal(defn.compile(fun, x, w, sc, fuse=True)(x, w, sc), defn.compile(fun, x, w, sc)(x, w, sc), "three calls")


# ---- stages over the same rows in one kernel (planned for compiled kernels) ------------------------------

def softmax_rows(x):
    z = Nx.multiply(x, 0.125)
    e = Nx.exp(Nx.subtract(z, Nx.reduce_max(z, axes=[-1], keep_axes=True)))
    return Nx.divide(e, Nx.sum(e, axes=[-1], keep_axes=True))


def centred_and_scaled(x, gain):  # layer-norm-like: mean, then mean of squares of the centred values
    n = x.shape[-1]
    mean = Nx.divide(Nx.sum(x, axes=[-1], keep_axes=True), float(n))
    c = Nx.subtract(x, mean)
    var = Nx.divide(Nx.sum(Nx.multiply(c, c), axes=[-1], keep_axes=True), float(n))
    return Nx.multiply(Nx.multiply(c, Nx.rsqrt(Nx.add(var, 1e-5))), gain)


def range_normalised(x):          # three statistics: minimum, maximum, and the sum of the result's numerator
    lo = Nx.reduce_min(x, axes=[-1], keep_axes=True)
    hi = Nx.reduce_max(x, axes=[-1], keep_axes=True)
    u = Nx.divide(Nx.subtract(x, lo), Nx.subtract(hi, lo))
    return Nx.divide(u, Nx.sum(u, axes=[-1], keep_axes=True))


def softmax_new_axis(x):          # statistics taken without keep_axes, then given their axis back
    m = Nx.new_axis(Nx.reduce_max(x, axes=[-1]), -1)
    e = Nx.exp(Nx.subtract(x, m))
    return Nx.divide(e, Nx.new_axis(Nx.sum(e, axes=[-1]), -1))


def log_softmax_rows(x):
    z = Nx.subtract(x, Nx.reduce_max(x, axes=[-1], keep_axes=True))
    return Nx.subtract(z, Nx.log(Nx.sum(Nx.exp(z), axes=[-1], keep_axes=True)))


def rms_scaled(x):                # one statistic, worked on with two constants and a square root; bf16 rounds at every node
    n = x.shape[-1]
    ms = Nx.divide(Nx.sum(Nx.multiply(x, x), axes=[-1], keep_axes=True), float(n))
    return Nx.divide(x, Nx.sqrt(Nx.add(ms, 1e-6)))


@pytest.mark.parametrize("ty", ["f32", "bf16"])
@pytest.mark.parametrize("shape", [(32, 512, 512), (100, 64), (7, 4096), (3, 5, 8), (1, 1024), (2049, 40)])
@pytest.mark.parametrize("name", ["softmax_rows", "centred_and_scaled", "range_normalised", "log_softmax_rows", "rms_scaled",
                                  "softmax_new_axis"])
def test_row_stages_are_bit_identical_to_node_by_node(name, shape, ty, hip):
    rng = np.random.default_rng(seed_of(name, shape, ty))
    x = rand_float(rng, ty, shape, hip)
    args = (x, rand_float(rng, ty, (shape[-1],), hip)) if name == "centred_and_scaled" else (x,)
    fun = {"softmax_rows": softmax_rows, "centred_and_scaled": centred_and_scaled, "range_normalised": range_normalised,
           "log_softmax_rows": log_softmax_rows, "rms_scaled": rms_scaled, "softmax_new_axis": softmax_new_axis}[name]
    want = defn.compile(fun, *args)(*args)
    planned = defn.compile(fun, *args, fuse="compiled")
    # work on a statistic before it is used (the mean and the variance of the second function are divided by n,
    # the variance goes through an rsqrt) belongs to the stage that makes it
    staged = True
    assert (type(planned.roots[0].data.args[0]).__name__ == "_RowCluster") == staged
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        if "mode" in k:
            calls.append(1)
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        assert_bits_equal(planned(*args), want, f"{name} {shape} {ty}")
    finally:
        hip.fused_elementwise = classmethod(original)
    if staged:
        assert calls == [1]  # one launch for all stages


@pytest.mark.parametrize("ty", ["f32", "bf16"])
@pytest.mark.parametrize("shape", [(8, 8192), (64, 4104), (16, 32000), (3, 16384), (5, 16392)])
@pytest.mark.parametrize("name", ["softmax_rows", "centred_and_scaled", "log_sum_exp_rows"])
def test_long_rows_take_a_block_each(name, shape, ty, hip):
    rng = np.random.default_rng(seed_of(name, shape, ty))
    x = rand_float(rng, ty, shape, hip)
    args = (x, rand_float(rng, ty, (shape[-1],), hip)) if name == "centred_and_scaled" else (x,)
    fun = {"softmax_rows": softmax_rows, "centred_and_scaled": centred_and_scaled, "log_sum_exp_rows": log_sum_exp_rows}[name]
    want = defn.compile(fun, *args)(*args)
    planned = defn.compile(fun, *args, fuse="compiled")
    assert type(planned.roots[0].data.args[0]).__name__ == "_RowCluster"
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        if "mode" in k:
            calls.append(1)
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        assert_bits_equal(planned(*args), want, f"{name} {shape} {ty}")
    finally:
        hip.fused_elementwise = classmethod(original)
    assert calls == [1]


def bias_and_scale_per_row(x, bias):  # no reduction: a row and a value per row against ragged rows
    return Nx.multiply(Nx.exp(Nx.add(x, bias)), Nx.slice_along_axis(x, 0, 1, axis=len(x.shape) - 1))


def sum_of_squares(x):
    return Nx.sum(Nx.multiply(x, Nx.tanh(x)), axes=[-1])


# a lane per row (no vector, one, two; tails of every kind); 8, 16, 32 lanes with one vector each at most; a wave, a block: one
# vector more or less than whole trips, heads and tails of every length in turn from row to row
RAGGED_ROWS = [(37, 3), (41, 8), (257, 10), (70, 17), (33, 65), (9, 129), (9, 257), (9, 519), (3, 5, 1001), (8, 4097), (3, 32767), (1, 77)]


@pytest.mark.parametrize("ty", ["f32", "bf16"])
@pytest.mark.parametrize("shape", RAGGED_ROWS)
@pytest.mark.parametrize("name", ["softmax_rows", "centred_and_scaled", "log_softmax_rows", "log_sum_exp_rows", "sum_of_squares",
                                  "bias_and_scale_per_row"])
def test_rows_of_any_length_in_one_launch(name, shape, ty, hip):
    """The bits of the nodes one by one, and nothing written around the result."""
    rng = np.random.default_rng(seed_of(name, shape, ty, "ragged"))
    x = rand_float(rng, ty, shape, hip)
    with_row = name in ("centred_and_scaled", "bias_and_scale_per_row")
    args = (x, rand_float(rng, ty, (shape[-1],), hip)) if with_row else (x,)
    fun = globals()[name]
    planned = defn.compile(fun, *args, fuse="compiled")
    launches = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        out = original(cls, *a, **k)  # (a refusal raises: the nodes would run one by one)
        launches.append(k.get("mode"))
        return out
    hip.fused_elementwise = classmethod(counting)
    try:
        got = planned(*args)
    finally:
        hip.fused_elementwise = classmethod(original)
    assert launches == ["compiled"], launches
    assert_bits_equal(got, defn.compile(fun, *args)(*args), f"{name} {shape} {ty}")


@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(12, 10), (9, 100), (9, 185), (9, 1001), (3, 8191)])
def test_ragged_rows_at_any_address_leave_their_neighbours(shape, ty, hip):
    """Operands and results one element behind a vector boundary; rows of infinities, NaN and the lowest number."""
    from nx_amd import types as T
    from test_gpu_elementwise import encode
    rng = np.random.default_rng(seed_of(shape, ty, "address"))
    n, size = int(np.prod(shape)), T.size_bytes(T.normalize(ty))
    words = raw(rand_float(rng, ty, (n + 24,), hip)).copy()
    special = encode(np.array([np.inf, -np.inf, np.nan, -6.0e4 if ty == "f16" else -3.0e38, 0.0, -0.0]), ty)
    words[1:1 + special.size] = special
    words[1 + shape[-1]:1 + 2 * shape[-1]] = special[1]  # a row of -inf
    store = from_numpy(words, ty, hip)
    x = Nx.from_pointer(hip, Nx.Pointer(kind="local", address=Nx.to_pointer(store).address + size, data_size=n * size), ty, shape, keep=store)
    want = defn.compile(softmax_rows, x)(x)
    assert_bits_equal(defn.compile(softmax_rows, x, fuse="compiled")(x), want, f"{shape} {ty}")
    np.testing.assert_array_equal(raw(store).view(np.uint8), words.view(np.uint8))


def test_a_select_on_integers_reads_a_row_that_later_stages_hold(hip):
    """A SELECT marked as an integer instruction takes its operands as floats all the same: the stage it stands in is the
    first that reads the row, and the registers that hold the row for the later stages are filled there."""
    from nx_amd.tensor import template
    SET, BINARY, SELECT, AS_TYPE, ROW_REDUCE, ROW_STAT = 0, 2, 3, 4, 6, 7
    CONST, INPUT, ROWSTAT, ADD, SUM, INT = 0, 1, 3, 0, 0, 2
    f32, s32 = ("f", 32), ("s", 32)
    program = [dict(kind=SET, src=CONST, imm=1.0, dt=f32), dict(kind=SELECT, src=INPUT, arg=0, src2=INPUT, arg2=0, flags=INT, dt=s32),
               dict(kind=AS_TYPE, dt=f32), dict(kind=ROW_REDUCE, op=SUM, dt=f32), dict(kind=ROW_STAT, arg=0, dt=f32),
               dict(kind=SET, src=INPUT, arg=0, dt=f32), dict(kind=BINARY, op=ADD, src=ROWSTAT, arg=0, dt=f32),
               dict(kind=ROW_REDUCE, op=SUM, dt=f32), dict(kind=ROW_STAT, arg=1, dt=f32),
               dict(kind=SET, src=INPUT, arg=0, dt=f32), dict(kind=BINARY, op=ADD, src=ROWSTAT, arg=1, dt=f32)]
    for rows, cols in ((9, 8), (5, 1024), (3, 4104)):
        x = np.random.default_rng(cols).integers(-3, 4, size=(rows, cols)).astype(np.float32)  # (every sum below 2^24: exact)
        got = hip.fused_elementwise(template("f32", (rows, cols)), program, [from_numpy(x, "f32", hip)], (rows, cols, [(cols, 1)]), mode="compiled")
        total = x.sum(axis=1, keepdims=True, dtype=np.float64)
        np.testing.assert_array_equal(hip.to_numpy(got), (x + (total + cols * total)).astype(np.float32))


# one vector a lane, two, three, eight; a block per row: three, eight, nine, sixteen, more than are held
@pytest.mark.parametrize("ty", ["f32", "bf16"])
@pytest.mark.parametrize("warmed,others", [((40, 64), [(9, 8), (9, 512), (5, 520), (7, 1024), (5, 1032), (3, 1544), (2049, 4096)]),
                                           ((3, 4104), [(5, 16384), (3, 16392), (8, 32760), (2048, 32776)])])
def test_a_program_that_holds_its_row_is_captured_at_other_lengths(warmed, others, ty, hip):
    """Rows of one length were run, rows of another are met in a capture: the program is there in a form that takes any
    length, nothing is compiled, and the bits are those of the nodes one by one."""
    from nx_amd import backend as B
    shift = {"f32": 0.37, "bf16": 0.375}[ty]  # (a constant no other test uses: a program of this test's own)

    def fun(x):
        z = Nx.subtract(Nx.add(x, shift), Nx.reduce_max(x, axes=[-1], keep_axes=True))
        return Nx.subtract(z, Nx.log(Nx.sum(Nx.exp(z), axes=[-1], keep_axes=True)))
    rng = np.random.default_rng(seed_of(warmed, ty, "one compilation"))
    before = B.fused_compiled_count()
    first = rand_float(rng, ty, warmed, hip)
    assert_bits_equal(defn.compile(fun, first, fuse="compiled")(first), defn.compile(fun, first)(first), f"{warmed}")
    assert B.fused_compiled_count() == before + 1
    for shape in others:
        x = rand_float(rng, ty, shape, hip)
        want = defn.compile(fun, x)(x)
        planned = defn.compile(fun, x, fuse="compiled")
        cluster = planned.roots[0].data.args[0]
        assert type(cluster).__name__ == "_RowCluster" and not any(ins.get("src") == 4 for ins in cluster.program)
        launches = []
        original = hip.fused_elementwise.__func__

        def counting(cls, *a, **k):
            out = original(cls, *a, **k)  # (a refusal raises: the nodes would run one by one)
            launches.append(k.get("mode"))
            return out
        hip.fused_elementwise = classmethod(counting)
        B.capture_begin(0)
        try:
            out = planned(x)
        finally:
            graph = B.capture_end(0)
            hip.fused_elementwise = classmethod(original)
        assert launches == ["compiled"] and B.fused_compiled_count() == before + 1, shape
        for _ in range(3):
            graph.launch()
            assert_bits_equal(out, want, f"replay at {shape}")
            assert_bits_equal(Nx.exp(x), Nx.exp(x), "work between the replays")
        del out
        graph.destroy()
    for shape in others:  # and outside a capture each length has kernels of its own
        x = rand_float(rng, ty, shape, hip)
        assert_bits_equal(defn.compile(fun, x, fuse="compiled")(x), defn.compile(fun, x)(x), f"{shape}")


# Functions with a branch, long ones and short ones on either side of where a program's trips are written out: one, two, four
# vectors a lane; a block per row with four, fifteen (values carried in a loop) and sixteen
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(9, 512), (9, 1024), (5, 2048), (3, 8192), (3, 30720), (2, 32000)])
@pytest.mark.parametrize("name", ["tanh", "sin", "pow", "atan2", "log"])
def test_row_stages_of_costly_functions_are_bit_identical(name, shape, ty, hip):
    function = {"pow": lambda x: Nx.pow(Nx.add(Nx.abs(x), 0.5), 1.25), "atan2": lambda x: Nx.atan2(x, 0.75),
                "log": lambda x: Nx.log(Nx.add(Nx.abs(x), 1.0))}.get(name, getattr(Nx, name, None))

    def held(x):  # the function again in every stage
        z = function(x)
        return Nx.subtract(z, Nx.log(Nx.sum(Nx.exp(Nx.subtract(z, Nx.reduce_max(z, axes=[-1], keep_axes=True))), axes=[-1], keep_axes=True)))

    def carried(x):
        z = function(x)
        return Nx.divide(z, Nx.add(Nx.sum(z, axes=[-1], keep_axes=True), 2.0))
    x = rand_float(np.random.default_rng(seed_of(name, shape, ty)), ty, shape, hip)
    for fun in (held, carried):
        planned = defn.compile(fun, x, fuse="compiled")
        assert type(planned.roots[0].data.args[0]).__name__ == "_RowCluster"
        assert_bits_equal(planned(x), defn.compile(fun, x)(x), f"{name} {shape} {ty}")


def test_rows_too_long_for_carried_values_are_read_again(hip):
    x = rand_float(np.random.default_rng(7), "f32", (2048, 32776), hip)
    planned = defn.compile(softmax_rows, x, fuse="compiled")
    cluster = planned.roots[0].data.args[0]
    assert type(cluster).__name__ == "_RowCluster" and not any(ins.get("src") == 4 for ins in cluster.program)
    assert_bits_equal(planned(x), defn.compile(softmax_rows, x)(x), "rows of 32776")


def test_rows_that_the_reduction_would_split_run_stage_by_stage(hip):
    x = rand_float(np.random.default_rng(6), "f32", (4, 65536), hip)   # few rows, very long: the separate sum works in segments
    planned = defn.compile(softmax_rows, x, fuse="compiled")
    assert_bits_equal(planned(x), defn.compile(softmax_rows, x)(x), "split rows")


def test_a_few_very_long_rows_keep_their_reduction_in_the_group(hip):
    """exp(t) / sum(exp(t)) over a million values (exla/bench/softmax.exs:1-41): the sum is cut into segments as the
    separate reduction cuts it, so the group that feeds it still holds it -- one call, the same bits -- and the
    refusal of the stage program, which the shape alone decides, is asked for once."""
    from nx_amd.backend import fused_mode as set_mode
    t = rand_float(np.random.default_rng(1000000), "f32", (1000000,), hip)

    def softmax(n):
        return Nx.divide(Nx.exp(n), Nx.sum(Nx.exp(n)))
    want = defn.compile(softmax, t)(t)
    planned = defn.compile(softmax, t, fuse="compiled")
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        calls.append(a[4] if len(a) > 4 else k.get("reduce_op", -1))
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        set_mode("compiled")
        assert_bits_equal(planned(t), want, "first call")
        first = list(calls)
        del calls[:]
        assert_bits_equal(planned(t), want, "second call")
        assert calls == [0, -1], calls            # the sum inside its group, then the quotient
        assert first in ([-1, 0, -1], [0, -1])    # (with the stage program offered and refused once, where one was planned)
    finally:
        set_mode("interpreted")
        hip.fused_elementwise = classmethod(original)


def test_configuration_3_softmax_in_one_kernel(hip):
    args = build_args(hip)["softmax"]
    planned = defn.compile(CHAINS["softmax"], *args, fuse="compiled")
    assert type(planned.roots[0].data.args[0]).__name__ == "_RowCluster"
    assert_bits_equal(planned(*args), defn.compile(CHAINS["softmax"], *args)(*args), "softmax of the scores")


def log_sum_exp_rows(x):
    m = Nx.reduce_max(x, axes=[-1], keep_axes=True)
    return Nx.add(Nx.log(Nx.sum(Nx.exp(Nx.subtract(x, m)), axes=[-1], keep_axes=True)), m)


def mean_rows(x):
    return Nx.mean(x, axes=[-1], keep_axes=True)


def root_mean_square_rows(x):
    return Nx.sqrt(Nx.divide(Nx.sum(Nx.multiply(x, x), axes=[-1], keep_axes=True), float(x.shape[-1])))


def spread_rows(x):               # the result reads two other statistics
    lo = Nx.reduce_min(x, axes=[-1], keep_axes=True)
    hi = Nx.reduce_max(x, axes=[-1], keep_axes=True)
    return Nx.divide(Nx.sum(Nx.subtract(x, lo), axes=[-1], keep_axes=True), hi)


def sum_of_a_masked_product(x, y):
    return Nx.sum(Nx.multiply(Nx.add(x, y), Nx.greater(x, 0.0)), axes=[1])


def largest_masked_product(x, y):
    return Nx.reduce_max(Nx.multiply(Nx.less_equal(y, 0.5), Nx.exp(x)), axes=[1], keep_axes=True)


def masked_softmax_rows(x, y):      # one mask is made by the stages, of the row they read, the other is an operand of theirs
    z = Nx.multiply(x, 0.125)
    e = Nx.multiply(Nx.exp(Nx.subtract(z, Nx.reduce_max(z, axes=[-1], keep_axes=True))), Nx.greater(x, 0.0))
    return Nx.multiply(Nx.greater(y, -1.0), Nx.divide(e, Nx.sum(e, axes=[-1], keep_axes=True)))


# rows of whole vectors and ragged ones, one to a wave and one to a block; numbers that are not finite under the mask
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(64, 256), (9, 185), (1, 7), (5, 8200), (2049, 40)])
@pytest.mark.parametrize("name", ["sum_of_a_masked_product", "largest_masked_product", "masked_softmax_rows"])
def test_values_times_a_mask_feed_reductions_and_row_stages(name, shape, ty, hip):
    fun = globals()[name]
    rng = np.random.default_rng(seed_of(name, shape, ty, "mask"))
    for make in (rand_float, not_finite):
        args = (make(rng, ty, shape, hip), make(rng, ty, shape, hip))
        planned = defn.compile(fun, *args, fuse="compiled")
        group = planned.roots[0].data.args[0]
        assert any(i["dt"] == ("u", 8) for i in group.program) and (type(group).__name__ == "_RowCluster" or group.reduce is not None)
        assert_bits_equal(planned(*args), defn.compile(fun, *args)(*args), f"{name} {shape} {ty}")


@pytest.mark.parametrize("ty", ["f32", "bf16"])
@pytest.mark.parametrize("shape", [(32, 512, 512), (100, 64), (7, 4096), (3, 5, 8), (1, 1024), (2049, 40)])
@pytest.mark.parametrize("name", ["log_sum_exp_rows", "mean_rows", "root_mean_square_rows", "spread_rows"])
def test_per_row_results_from_one_kernel_are_bit_identical(name, shape, ty, hip):
    rng = np.random.default_rng(seed_of(name, shape, ty))
    x = rand_float(rng, ty, shape, hip)
    fun = {"log_sum_exp_rows": log_sum_exp_rows, "mean_rows": mean_rows, "root_mean_square_rows": root_mean_square_rows,
           "spread_rows": spread_rows}[name]
    want = defn.compile(fun, x)(x)
    planned = defn.compile(fun, x, fuse="compiled")
    cluster = planned.roots[0].data.args[0]
    assert type(cluster).__name__ == "_RowCluster" and cluster.program[-1].get("flags") == 1
    calls = []
    original = hip.fused_elementwise.__func__

    def counting(cls, *a, **k):
        if "mode" in k:
            calls.append(1)
        return original(cls, *a, **k)
    hip.fused_elementwise = classmethod(counting)
    try:
        assert_bits_equal(planned(x), want, f"{name} {shape} {ty}")
    finally:
        hip.fused_elementwise = classmethod(original)
    assert calls == [1]


# ---- a flat index space that is no whole number of vectors (compiled groups take the partial last one) ----

@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(1,), (7,), (9,), (37, 11), (3, 5, 7), (1000003,), (255, 257)])
def test_ragged_sizes_in_compiled_groups(shape, ty, hip):
    rng = np.random.default_rng(seed_of(shape, ty))
    x, y = rand_float(rng, ty, shape, hip), rand_float(rng, ty, shape, hip)
    guard = rand_float(rng, ty, (64,), hip)   # a neighbour in memory that must stay as it is

    def fun(a, b):
        h = Nx.add(Nx.multiply(a, 0.5), b)
        return Nx.select(Nx.greater(h, 0.0), Nx.tanh(h), Nx.multiply(h, 0.01))

    want = defn.compile(fun, x, y)(x, y)
    before = hip.to_numpy(guard).copy()
    planned = defn.compile(fun, x, y, fuse="compiled")
    assert planned.roots[0].data.op == "fused" and planned.roots[0].data.args[0].layout is not None
    assert_bits_equal(planned(x, y), want, f"ragged {shape} {ty}")
    np.testing.assert_array_equal(hip.to_numpy(guard), before)
    # planned without the compiled kernels in mind, such a shape is left to the separate callbacks
    assert_bits_equal(defn.compile(fun, x, y, fuse=True)(x, y), want, f"ragged {shape} {ty}, mode-agnostic plan")


def test_ragged_integer_words(hip):
    x = rand_words(np.random.default_rng(12), "u32", (1001,), hip)
    planned = defn.compile(bits_to_unit_floats, x, fuse="compiled")
    assert planned.roots[0].data.op == "fused"
    assert_bits_equal(planned(x), defn.compile(bits_to_unit_floats, x)(x), "ragged u32 -> f32")


def test_ragged_rows_still_fall_back(hip):
    rng = np.random.default_rng(13)
    x, bias = rand_float(rng, "f32", (37, 11), hip), rand_float(rng, "f32", (11,), hip)   # a row operand: no flat index space

    def fun(a, b):
        return Nx.exp(Nx.add(a, b))
    planned = defn.compile(fun, x, bias, fuse="compiled")
    assert_bits_equal(planned(x, bias), defn.compile(fun, x, bias)(x, bias), "row operand, ragged rows")


@pytest.mark.parametrize("ty", ["f16", "bf16", "f32"])
def test_fused_groups_on_special_values(ty, hip):
    """Every unary and binary element-wise node a group can hold, on zeros of either sign, the smallest numbers, domain
    ends, infinities and NaN: the group's bits are those of the nodes run one by one, interpreted and compiled."""
    from nx_amd.backend import fused_mode as set_mode
    from test_gpu_elementwise import MATH, encode
    tiny = {"f16": 6e-8, "bf16": 1e-38, "f32": 1e-45}[ty]
    large = 8.0 if ty == "f16" else 30.0
    v = np.array([0.0, -0.0, tiny, -tiny, 1.0, -1.0, 0.5, -0.5, 2.0, -2.0, np.inf, -np.inf, np.nan, 1e-4, -1e-4, large, -large,
                  3.0, -3.0, 0.25, -0.25, 1.5, -1.5, 7.0])
    x = from_numpy(encode(v, ty), ty, hip)
    a, b = [g.ravel() for g in np.meshgrid(v[:16], v[:16], indexing="ij")]
    ha, hb = from_numpy(encode(a, ty), ty, hip), from_numpy(encode(b, ty), ty, hip)
    programs = [(f"{op} then negate", (lambda t, op=op: Nx.negate(getattr(Nx, op)(t))), (x,)) for op in MATH]
    programs += [(f"{op} plus its operand", (lambda t, op=op: Nx.add(getattr(Nx, op)(t), t)), (x,)) for op in MATH]
    programs += [(f"{op} then negate", (lambda p, q, op=op: Nx.negate(getattr(Nx, op)(p, q))), (ha, hb))
                 for op in ("add", "subtract", "multiply", "divide", "pow", "atan2", "min", "max")]
    programs += [(f"{op} times its operand", (lambda p, q, op=op: Nx.multiply(getattr(Nx, op)(p, q), q)), (ha, hb))
                 for op in ("add", "subtract", "multiply", "divide", "min", "max")]
    try:
        for name, fun, args in programs:
            want = defn.compile(fun, *args)(*args)
            for mode in ("interpreted", "compiled"):
                set_mode(mode)
                assert_bits_equal(defn.compile(fun, *args, fuse=True)(*args), want, f"{name}, {ty}, {mode}")
    finally:
        set_mode("interpreted")


def split_heads(t, heads):
    return Nx.transpose(Nx.reshape(t, (t.shape[0], t.shape[1], heads, t.shape[2] // heads)), axes=[0, 2, 1, 3])


# scores of heads split off projected activations: whole and partial slabs of K, one query (decoding), odd numbers of keys, every
# kernel the tile choice can come to; K that is not whole 16-byte pieces is copied as before
@pytest.mark.parametrize("ty", ["bf16", "f16", "f32", "s8"])
@pytest.mark.parametrize("batch,heads,queries,keys,dim", [(2, 3, 40, 72, 64), (1, 4, 1, 333, 128), (3, 2, 130, 257, 72), (2, 8, 256, 512, 64),
                                                          (1, 2, 512, 640, 1024), (2, 2, 17, 65, 33), (1, 1, 24, 48, 64),
                                                          (2, 3, 16, 24, 4096), (1, 2, 1, 300, 1024), (2, 2, 4, 64, 2048)])
def test_a_dot_reads_transposed_operands_where_they_lie(batch, heads, queries, keys, dim, ty, hip):
    rng = np.random.default_rng(seed_of(batch, heads, queries, keys, dim, ty))

    def rand(*shape):
        if ty == "s8":
            return from_numpy(rng.integers(-99, 100, size=shape).astype(np.int8), "s8", hip)
        return rand_float(rng, ty, shape, hip)
    q, k, p = rand(batch, queries, heads * dim), rand(batch, keys, heads * dim), rand(batch, heads, queries, keys)
    out = {"out_type": "s32"} if ty == "s8" else {}

    def scores(a, b):
        return Nx.dot(split_heads(a, heads), [3], [0, 1], split_heads(b, heads), [3], [0, 1], **out)

    def mixed(a, b):  # the right operand K-outer, where it lies (the values of an attention)
        return Nx.dot(a, [3], [0, 1], split_heads(b, heads), [2], [0, 1], **out)
    copies = []
    original = hip.transpose.__func__

    def counting(cls, *a, **kw):
        copies.append(1)
        return original(cls, *a, **kw)
    for fun, args, row_block in ((scores, (q, k), 1), (mixed, (p, k), {"bf16": 8, "f16": 8, "f32": 4, "s8": 16}[ty])):
        want = defn.compile(fun, *args)(*args)
        planned = defn.compile(fun, *args, fuse="compiled")
        assert planned.roots[0].data.op == "dot_views"
        copies.clear()
        hip.transpose = classmethod(counting)
        try:
            got = planned(*args)
        finally:
            hip.transpose = classmethod(original)
        assert_bits_equal(got, want, f"{fun.__name__} {ty}")
        esz, K = {"s8": 1, "f32": 4}.get(ty, 2), dim if fun is scores else keys
        direct = K * esz % 16 == 0 and (fun is scores or dim % row_block == 0) and queries * (keys if fun is scores else dim) >= 256
        if (queries <= 32 and keys <= 32 and K >= 4096) or (fun is scores and esz == 4 and queries <= 4 and K >= 1024):
            direct = False  # (few outputs over a long K are summed in f64 -- s8 exactly -- by the separate contraction)
        assert (not copies) == direct, (fun.__name__, ty, copies)


def test_other_orders_of_a_dots_operands(hip, oracle):
    """Operands whose kept or contracted axes are not neighbours, batch axes in two orders, a transposed operand with a second reader."""
    rng = np.random.default_rng(77)
    a, b = rand_float(rng, "bf16", (4, 32, 6, 64), hip), rand_float(rng, "bf16", (6, 4, 48, 64), hip)

    def apart(x, y):          # kept axes (0, 2) of x are not neighbours in memory once 1 is contracted with 3
        return Nx.dot(Nx.transpose(x, axes=[1, 3, 0, 2]), [0, 1], Nx.reshape(Nx.transpose(y, axes=[3, 0, 1, 2]), (32, 64, 36)), [0, 1])

    def batched(x, y):        # batch axes in another order on either side
        return Nx.dot(Nx.transpose(x, axes=[0, 2, 1, 3]), [3], [0, 1], Nx.transpose(y, axes=[1, 0, 2, 3]), [3], [0, 1])

    def read_twice(x, y):
        t = Nx.transpose(x, axes=[0, 2, 1, 3])
        return Nx.add(Nx.dot(t, [3], [0, 1], Nx.transpose(y, axes=[1, 0, 2, 3]), [3], [0, 1]), Nx.sum(t))
    for fun in (apart, batched, read_twice):
        assert_bits_equal(defn.compile(fun, a, b, fuse="compiled")(a, b), defn.compile(fun, a, b)(a, b), fun.__name__)


def test_dot_strided_refuses_what_is_not_there(hip):
    """Strides that reach past an operand's end, overlapping rows, extents below zero: an error, and nothing is launched."""
    import ctypes as C

    from nx_amd import backend as B
    from nx_amd.backend import K_INNER
    x = rand_float(np.random.default_rng(1), "bf16", (4, 32, 64), hip)
    out = rand_float(np.random.default_rng(2), "bf16", (4, 32, 32), hip)
    good = (0, 32 * 64, 64)

    def call(ls, rs, K=64, M=32, outer=1, inner=4):
        return L.lib.hipnx_dot_strided(_Context.get(0), T_BF16, T_BF16, T_BF16, outer, inner, M, 32, K, K_INNER, K_INNER,
                                       L.i64_array(ls), L.i64_array(rs), x.data.ref.handle, x.data.ref.handle, out.data.ref.handle)
    from nx_amd import types as T
    T_BF16 = T.code(("bf", 16))
    assert call(good, good) == 0
    for bad in ((0, 32 * 64 + 8, 64), (0, 32 * 64, 72), (8, 32 * 64, 64), (0, 32 * 64, 56), (0, -64, 64), (0, 32 * 64, 1 << 41)):
        assert call(bad, good, outer=2 if bad[0] else 1, inner=4) != 0 and call(good, bad, outer=2 if bad[0] else 1) != 0, bad
    assert call(good, good, M=-1) != 0 and call(good, good, K=72) != 0
    # products that are small numbers, or none, in 64 bits: rows 2^40 elements apart, batches of 2^62 items
    for M, stride in (((1 << 23) + 1, 1 << 40), ((1 << 24) + 1, 1 << 40), ((1 << 25) + 1, 1 << 39), ((1 << 60) + 1, 64), ((1 << 59) + 1, 64)):
        for inner in (1, 4):
            assert call((0, 32 * 64, stride), good, M=M, inner=inner) == L.EINVAL and "dot_strided lhs" in L.last_error(), (M, stride)
    assert call((1 << 40, 0, 64), good, outer=(1 << 24) + 1, inner=1) != 0 and call(good, (0, 1 << 40, 64), inner=(1 << 23) + 1) != 0
    assert call(good, good, outer=1 << 32, inner=1 << 31) != 0
    for shape in ((1 << 31, 1 << 33, 64), (1 << 62, 4, 8), (4, 1 << 62, 8), (32, 32, 1 << 61)):
        assert L.lib.hipnx_dot(_Context.get(0), T_BF16, T_BF16, T_BF16, 1, *shape, K_INNER, K_INNER, x.data.ref.handle, x.data.ref.handle,
                               out.data.ref.handle) == L.EINVAL, shape
    row_reduce, row_stat = L.FUSED_BITCAST + 1, L.FUSED_BITCAST + 2
    instr = (L.FusedInstr * 3)()
    for q, (kind, op, src) in zip(instr, ((L.FUSED_SET, 0, L.FUSED_SRC_INPUT), (row_reduce, 0, 0), (row_stat, 0, 0))):
        q.kind, q.op, q.src, q.dt, q.flags = kind, op, src, T.code(("f", 32)), kind == row_stat

    def scores(M, l, r):
        handles = (C.c_void_p * 1)(x.data.ref.handle)
        return L.lib.hipnx_fused_scores(_Context.get(0), 3, C.cast(instr, C.c_void_p), 1, handles, (C.c_int * 1)(T_BF16), (C.c_int64 * 1)(32), (C.c_int * 1)(1),
                                        32, 0, 1, 4, M, 64, (C.c_int64 * 6)(*l, *r), (C.c_void_p * 2)(x.data.ref.handle, x.data.ref.handle),
                                        T.code(("f", 32)), out.data.ref.handle)
    B._set_fused_mode("compiled", 0)
    try:
        assert scores(32, good, good) == 0
        for M, stride in (((1 << 23) + 1, 1 << 40), ((1 << 24) + 1, 1 << 40), ((1 << 25) + 1, 1 << 39)):
            assert scores(M, (0, 32 * 64, stride), good) == L.EINVAL and "fused_scores lhs" in L.last_error(), (M, stride)
    finally:
        B._set_fused_mode("interpreted", 0)


# ---- traced functions and callbacks issued natively (nx_amd/replay.py, csrc/calls.c) ----------------------

def replayed_functions(hip):
    rng = np.random.default_rng(99)

    def r(*shape, ty="f32"):
        return lambda: rand_float(rng, ty, shape, hip)

    def words(*shape):
        return lambda: from_numpy(rng.integers(0, 2 ** 32, size=shape, dtype=np.uint32), "u32", hip)

    def normalised(x, g):
        return centred_and_scaled(x, g), Nx.sum(x, axes=[0]), Nx.add(Nx.multiply(x, 0.5), 3)

    def step(x, w, b):
        h = Nx.max(Nx.add(Nx.dot(x, w), b), 0.0)
        return Nx.subtract(w, Nx.multiply(Nx.dot(x, [0], h, [0]), 0.1)), Nx.mean(h)

    def moved(x):
        return Nx.concatenate([Nx.reverse(x, axes=[1]), Nx.transpose(Nx.transpose(x))], axis=0), Nx.slice_along_axis(x, 1, 2, axis=1), Nx.select(Nx.greater(x, 0.0), x, 0.0)

    def picked(x, t):
        best = Nx.argmax(x, axis=1, type="u32")
        return best, Nx.take(t, best)
    return {"normalised": (normalised, [r(9, 24), r(24)]), "softmax": (softmax_rows, [r(6, 33, ty="bf16")]), "step": (step, [r(16, 24), r(24, 40), r(40)]),
            "moved": (moved, [r(5, 8)]), "picked": (picked, [r(7, 50), r(50, 16, ty="bf16")]),
            "normal": (lambda k: Random.normal(k, shape=(1001,))[0], [words(2)])}


@pytest.mark.parametrize("name", ["normalised", "softmax", "step", "moved", "picked", "normal"])
def test_a_recorded_function_gives_each_call_its_own_results(name, hip):
    """Every call after the recording on operands of its own, earlier results kept, dropped and deallocated in between: the
    bits of the nodes one by one, results in buffers of their own, and no memory that stays behind."""
    fun, makers = replayed_functions(hip)[name]
    planned = defn.compile(fun, *[m() for m in makers], fuse="compiled")
    plain = defn.compile(fun, *[m() for m in makers])
    kept, wanted = [], []
    for i in range(9):
        args = [m() for m in makers]
        want = plain._walk(args)
        got = planned._evaluate(args)
        for g, w in zip(got, want):
            assert_bits_equal(g, w, f"{name}, call {i}")
        kept.append(got)
        wanted.append(want)
        if i == 5:
            for t in kept.pop(0):
                assert Nx.backend_deallocate(t) == "ok" and Nx.backend_deallocate(t) == "already_deallocated"
            wanted.pop(0)
    assert planned.replay is not None, "not recorded"
    for got, want in zip(kept, wanted):
        for g, w in zip(got, want):
            assert_bits_equal(g, w, f"{name}, kept")
    assert len({Nx.to_pointer(t).address for got in kept for t in got}) == sum(len(got) for got in kept)
    args = [m() for m in makers]
    del kept, wanted, got, want, g, w
    gc.collect()
    planned._evaluate(args)
    before = mem_stats()["live"]
    for _ in range(5):
        planned._evaluate(args)
    assert mem_stats()["live"] == before


def test_a_recording_is_left_where_it_does_not_apply(hip):
    from nx_amd import HostBinary
    from nx_amd import backend as B

    def fun(x, t):
        return Nx.as_type(x, "bf16"), Nx.take(t, Nx.as_type(Nx.reduce_max(x, axes=[1]), "s32"))
    x = from_numpy(np.arange(12, dtype=np.float32).reshape(3, 4) / 4 + 0.1234, "f32", hip)
    t = rand_float(np.random.default_rng(3), "f32", (4, 8), hip)
    planned, plain = defn.compile(fun, x, t, fuse="compiled"), defn.compile(fun, x, t)
    for _ in range(5):
        planned(x, t)
    assert planned.replay is not None

    def same(*args):
        for g, w in zip(planned._evaluate(list(args)), plain._walk(list(args))):
            assert_bits_equal(g, w, "")
    same(x, t)
    previous = B.bf16_rounding("nearest_even")     # a setting the calls were laid out under
    try:
        same(x, t)
    finally:
        B.bf16_rounding(previous)
    same(x, Nx.backend_copy(t, HostBinary, {}))   # an operand elsewhere
    far = from_numpy(np.full((3, 4), 77.0, dtype=np.float32), "f32", hip)
    for _ in range(2):                              # what the library refuses is reported as ever
        with pytest.raises(Exception, match="index 77 is out of bounds"):
            planned(far, t)
    previous = B.bounds_policy("clamp")
    try:
        same(far, t)
    finally:
        B.bounds_policy(previous)
    gone = Nx.backend_copy(x, hip, {"device": 0})
    Nx.backend_deallocate(gone)
    with pytest.raises(L.HipNxError):
        planned(gone, t)
    same(x, t)
    with pytest.raises(ValueError):
        planned(t, x)


@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("cols", [10, 72, 185, 512, 1001])
def test_quotients_of_exponentials_are_divisions(cols, ty, hip):
    """exp(x) / s over rows whose exponentials lie on both sides of every bound of the quick quotient: zeros, subnormal numbers,
    infinities, NaN; divisors of all sizes."""
    rng = np.random.default_rng(seed_of(cols, ty, "quotients"))
    span = {"f16": 9.0, "bf16": 100.0, "f32": 104.0}[ty]
    x = rng.uniform(-span, 0, (64, cols)).astype(np.float32)
    x[:16] = rng.uniform(-3, 3, (16, cols))
    x[16:24, ::3] = -np.inf
    x[24:28, 1::5] = 60.0 if ty != "f16" else 9.0
    x[28:30, 2::7], x[30, 3], x[31, 4] = 80.0 if ty != "f16" else 10.0, np.inf, np.nan
    scale = np.float32(2.0) ** rng.integers(-60, 60, (64, 1)).astype(np.float32) * rng.uniform(1, 2, (64, 1)).astype(np.float32)
    s = from_numpy(scale, "f32", hip)
    t = from_numpy((x.view(np.uint32) >> 16).astype(np.uint16) if ty == "bf16" else x.astype(np.float16 if ty == "f16" else np.float32), ty, hip)

    def softmaxed(v):
        e = Nx.exp(v)
        return Nx.divide(e, Nx.sum(e, axes=[-1], keep_axes=True))

    def scaled(v, w):  # the divisor's size set by an operand
        e = Nx.exp(Nx.as_type(v, "f32"))
        return Nx.divide(e, Nx.multiply(Nx.sum(Nx.multiply(e, w), axes=[-1], keep_axes=True), 0.37))
    for fun, args in ((softmaxed, (t,)), (scaled, (t, s))):
        assert_bits_equal(defn.compile(fun, *args, fuse="compiled")(*args), defn.compile(fun, *args)(*args), f"{fun.__name__} {cols} {ty}")


def test_what_cannot_be_recorded_is_evaluated(hip):
    """One buffer under two parameters when the recording would be made, parameters and constants handed through, one buffer
    under two results, control flow."""
    x = rand_float(np.random.default_rng(5), "f32", (4, 8), hip)
    y = rand_float(np.random.default_rng(6), "f32", (4, 8), hip)
    twice = defn.compile(lambda a, b: Nx.subtract(Nx.multiply(a, 2.0), b), x, y, fuse="compiled")
    for _ in range(5):
        twice(x, x)
    assert twice.replay is None
    assert_bits_equal(twice(x, y), Nx.subtract(Nx.multiply(x, 2.0), y), "other operands afterwards")
    for fun in (lambda a: (a, Nx.exp(a)), lambda a: (lambda e: (e, Nx.reshape(e, (32,))))(Nx.exp(a)),
                lambda a: defn.cond(Nx.greater(Nx.sum(a), 1.0e9), lambda: Nx.negate(a), lambda: Nx.exp(a))):
        planned, plain = defn.compile(fun, x), defn.compile(fun, x)
        for i in range(6):
            z = rand_float(np.random.default_rng(i), "f32", (4, 8), hip)
            for g, w in zip(planned._evaluate([z]), plain._walk([z])):
                assert_bits_equal(g, w, "")
        assert planned.replay is None


def test_recorded_functions_and_callbacks_from_several_threads(hip):
    import threading
    rng = np.random.default_rng(8)
    x, g = rand_float(rng, "f32", (33, 40), hip), rand_float(rng, "f32", (40,), hip)
    planned = defn.compile(centred_and_scaled, x, g, fuse="compiled")
    inputs = [rand_float(rng, "f32", (33, 40), hip) for _ in range(4)]
    wants = [defn.compile(centred_and_scaled, x, g)(i, g) for i in inputs]
    eager = [Nx.sum(Nx.exp(Nx.multiply(Nx.add(i, i), 0.5)), axes=[1]) for i in inputs]
    errors = []

    def work(k):
        try:
            for _ in range(40):  # (the recording happens while the others evaluate)
                assert_bits_equal(planned(inputs[k], g), wants[k], f"thread {k}")
                assert_bits_equal(Nx.sum(Nx.exp(Nx.multiply(Nx.add(inputs[k], inputs[k]), 0.5)), axes=[1]), eager[k], f"thread {k}, eager")
        except BaseException as e:  # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_callbacks_laid_out_once_follow_their_operands(hip):
    """The same signature again and again: numbers that change, operands elsewhere or gone, settings that change."""
    from nx_amd import backend as B
    x = rand_float(np.random.default_rng(1), "f32", (6, 10), hip)
    v = hip.to_numpy(x)
    for c in (0.5, -3.25, 0.0, -0.0, 7.0):
        np.testing.assert_array_equal(hip.to_numpy(Nx.multiply(x, c)).view(np.uint32), (v * np.float32(c)).view(np.uint32))
        np.testing.assert_array_equal(hip.to_numpy(Nx.add(x, int(c))), v + np.float32(int(c)))
    u = from_numpy(np.arange(60, dtype=np.uint8).reshape(6, 10), "u8", hip)
    assert Nx.add(u, 1).type == ("u", 8) and Nx.add(u, -1).type == ("s", 16) and Nx.add(u, 1.5).type == ("f", 32)
    gone = Nx.backend_copy(x, hip, {"device": 0})
    Nx.add(gone, x)
    Nx.backend_deallocate(gone)
    for call in (lambda: Nx.add(gone, x), lambda: Nx.exp(gone), lambda: Nx.sum(gone, axes=[1]), lambda: Nx.argmax(gone, axis=1), lambda: Nx.dot(gone, Nx.transpose(x))):
        with pytest.raises(L.HipNxError):
            call()
    t = rand_float(np.random.default_rng(2), "f32", (5, 4), hip)
    near, far = from_numpy(np.array([1, 4], np.int32), "s32", hip), from_numpy(np.array([1, 9], np.int32), "s32", hip)
    Nx.take(t, near)
    with pytest.raises(Exception, match="index 9 is out of bounds"):
        Nx.take(t, far)
    previous = B.bounds_policy("clamp")
    try:
        np.testing.assert_array_equal(hip.to_numpy(Nx.take(t, far)), hip.to_numpy(t)[[1, 4]])
    finally:
        B.bounds_policy(previous)
    b = from_numpy(np.array([[1.01, 1.0], [1.0, 1.0]], np.float32), "f32", hip)
    y = Nx.as_type(b, "bf16")
    for mode in ("truncate", "nearest_even", "truncate"):
        previous = B.bf16_rounding(mode)
        try:
            want = defn.compile(lambda p, q: Nx.dot(p, [1], q, [0]), y, y)._walk([y, y])[0]
            assert_bits_equal(Nx.dot(y, [1], y, [0]), want, mode)
        finally:
            B.bf16_rounding(previous)


def attention_probabilities(q, k, heads, mask=None, log=False):
    scores = Nx.dot(split_heads(q, heads), [3], [0, 1], split_heads(k, heads), [3], [0, 1])
    z = Nx.multiply(Nx.as_type(scores, "f32"), 0.125)
    if mask is not None:
        z = Nx.add(z, mask)
    return log_softmax_rows(z) if log else softmax_rows(z)


# one query row and rows around a block's sixteen; rows of columns in every form (whole vectors, 8 to 32 lanes, heads and tails),
# steps of 512 columns; K of one to eight steps
@pytest.mark.parametrize("ty", ["bf16", "f16"])
@pytest.mark.parametrize("batch,heads,queries,keys,dim", [(2, 3, 1, 320, 64), (3, 2, 16, 16, 32), (2, 2, 17, 100, 64), (1, 5, 33, 185, 128), (2, 4, 31, 512, 64),
                                                          (1, 3, 40, 513, 96), (2, 2, 64, 1001, 64), (1, 2, 20, 2041, 32), (14, 1, 300, 4096, 32), (4, 16, 18, 250, 256)])
def test_row_stages_contract_their_scores_themselves(batch, heads, queries, keys, dim, ty, hip):
    """On whole numbers, whose sums are exact in any order: the bits of the nodes one by one, and no contraction of its own."""
    rng = np.random.default_rng(seed_of(batch, heads, queries, keys, dim, ty))

    def whole(*shape):
        v = rng.integers(-2, 3, size=shape).astype(np.float32)
        return from_numpy((v.view(np.uint32) >> 16).astype(np.uint16) if ty == "bf16" else v.astype(np.float16), ty, hip)
    q, k = whole(batch, queries, heads * dim), whole(batch, keys, heads * dim)
    guard = whole(64)
    before = raw(guard).copy()
    mask = rand_float(rng, "f32", (batch, heads, queries, keys), hip)
    calls = []
    original = hip.fused_scores.__func__

    def counting(cls, *a, **kw):
        out = original(cls, *a, **kw)  # (a refusal raises)
        calls.append(1)
        return out
    for fun, args in ((lambda a, b: attention_probabilities(a, b, heads), (q, k)), (lambda a, b: attention_probabilities(a, b, heads, log=True), (q, k)),
                      (lambda a, b, m: attention_probabilities(a, b, heads, m), (q, k, mask))):
        planned = defn.compile(fun, *args, fuse="compiled")
        if len(args) == 3:  # (the masked scores are a tensor of their own: two full-size operands)
            assert_bits_equal(planned(*args), defn.compile(fun, *args)(*args), f"{ty}, mask")
            continue
        assert planned.roots[0].data.args[0].scores is not None
        calls.clear()
        hip.fused_scores = classmethod(counting)
        try:
            got = planned(*args)
        finally:
            hip.fused_scores = classmethod(original)
        assert calls == [1]
        assert_bits_equal(got, defn.compile(fun, *args)(*args), f"{ty}")
    np.testing.assert_array_equal(raw(guard), before)


@pytest.mark.parametrize("ty", ["bf16", "f16"])
def test_scores_that_are_left_to_the_contraction(ty, hip):
    """K off the steps of 32, few results per item (summed in f64 there), rows of more than 4096, one block per item over a large right
    operand, the other rounding: two calls, the same values as ever."""
    from nx_amd import backend as B
    rng = np.random.default_rng(seed_of(ty, "left"))
    for batch, heads, queries, keys, dim in ((2, 2, 20, 64, 40), (1, 4, 1, 100, 64), (1, 1, 8, 4104, 32), (1, 2, 1, 2048, 128)):
        q, k = rand_float(rng, ty, (batch, queries, heads * dim), hip), rand_float(rng, ty, (batch, keys, heads * dim), hip)
        fun = lambda a, b: attention_probabilities(a, b, heads)  # noqa: E731
        planned, want = defn.compile(fun, q, k, fuse="compiled"), defn.compile(fun, q, k)(q, k)
        for _ in range(4):
            assert_bits_equal(planned(q, k), want, f"{queries} x {keys} x {dim}")
        assert planned.replay is not None  # (a refusal does not keep the two calls from being recorded)
    q, k = rand_float(rng, ty, (2, 20, 128), hip), rand_float(rng, ty, (2, 64, 128), hip)
    fun = lambda a, b: attention_probabilities(a, b, 2)  # noqa: E731
    planned = defn.compile(fun, q, k, fuse="compiled")
    previous = B.bf16_rounding("nearest_even")
    try:
        assert_bits_equal(planned(q, k), defn.compile(fun, q, k)(q, k), "nearest even")
    finally:
        B.bf16_rounding(previous)


def test_a_dot_over_three_batch_axes(hip):
    """Batches that fold to two axes are read where they lie, others are copied: the same bits."""
    rng = np.random.default_rng(78)
    x, y = rand_float(rng, "bf16", (2, 3, 20, 4, 64), hip), rand_float(rng, "bf16", (2, 3, 24, 4, 64), hip)
    z, w = rand_float(rng, "f32", (3, 20, 2, 4, 32), hip), rand_float(rng, "f32", (4, 3, 2, 24, 32), hip)

    def heads_last(a, b):     # batch axes 0 and 1 are neighbours, the third lies behind the rows
        return Nx.dot(Nx.transpose(a, axes=[0, 1, 3, 2, 4]), [4], [0, 1, 2], Nx.transpose(b, axes=[0, 1, 3, 2, 4]), [4], [0, 1, 2])

    def all_apart(a, b):      # no two of them are neighbours in the same order on either side
        return Nx.dot(Nx.transpose(a, axes=[2, 0, 3, 1, 4]), [4], [0, 1, 2], Nx.transpose(b, axes=[2, 1, 0, 3, 4]), [4], [0, 1, 2])
    for fun, args in ((heads_last, (x, y)), (all_apart, (z, w))):
        planned = defn.compile(fun, *args, fuse="compiled")
        assert planned.roots[0].data.op == "dot_views"
        for _ in range(4):  # (the last one from its recording)
            assert_bits_equal(planned(*args), defn.compile(fun, *args)(*args), fun.__name__)
        assert planned.replay is not None


# both layouts on either side; rows, and items of the two batch axes, any number of elements apart
@pytest.mark.parametrize("ty", ["bf16", "f16", "f32", "s8"])
@pytest.mark.parametrize("layouts", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K,gap", [(32, 48, 64, 1), (144, 272, 128, 3), (272, 528, 208, 8), (64, 1040, 1072, 5)])
def test_strided_operands_lie_anywhere(M, N, K, gap, layouts, ty, hip):
    """Whole numbers, exact in any order.  What is between the rows is no operand: numbers that would show."""
    from nx_amd import types as T
    from nx_amd.backend import K_INNER, K_OUTER
    rng = np.random.default_rng(seed_of(M, N, K, gap, layouts, ty))
    outer, inner = 2, 3

    def operand(rows, k_inner):
        runs, run = (rows, K) if k_inner else (K, rows)
        ld = run + gap
        item = runs * ld + gap
        strides = (inner * item + gap, item, ld)
        v = np.full(outer * strides[0] + gap, 77.0, np.float32)
        values = rng.integers(-2, 3, size=(outer, inner, runs, run)).astype(np.float32)
        for o in range(outer):
            for i in range(inner):
                np.lib.stride_tricks.as_strided(v[o * strides[0] + i * item:], (runs, run), (4 * ld, 4))[:] = values[o, i]
        held = (v.view(np.uint32) >> 16).astype(np.uint16) if ty == "bf16" else v.astype({"f16": np.float16, "f32": np.float32, "s8": np.int8}[ty])
        return from_numpy(held, ty, hip), L.i64_array(strides), values if k_inner else values.transpose(0, 1, 3, 2), K_INNER if k_inner else K_OUTER
    l, ls, a, l_layout = operand(M, layouts[0] == "n")
    r, rs, b, r_layout = operand(N, layouts[1] == "t")
    ot = T.normalize("s32" if ty == "s8" else "f32")
    out = from_numpy(np.zeros((outer, inner, M, N), np.int32 if ty == "s8" else np.float32), ot, hip)
    code = T.code(T.normalize(ty))
    L.check(L.lib.hipnx_dot_strided(_Context.get(0), code, code, T.code(ot), outer, inner, M, N, K, l_layout, r_layout, ls, rs,
                                    l.data.ref.handle, r.data.ref.handle, out.data.ref.handle))
    np.testing.assert_array_equal(hip.to_numpy(out).astype(np.float64), a.astype(np.float64) @ b.astype(np.float64).transpose(0, 1, 3, 2))


@pytest.mark.parametrize("fuse", [False, True, "compiled"])
def test_a_recorded_function_tells_its_numbers_from_its_arguments(fuse, hip):
    """A rate given as an argument, equal to a number of the function while it is recorded."""
    x = rand_float(np.random.default_rng(4), "f32", (12, 16), hip)

    def fun(t, rate):
        return Nx.subtract(t, Nx.multiply(Nx.exp(t), rate)), Nx.add(t, 0.5), Nx.max(t, rate)
    previous = Nx.default_backend(hip)  # (where numbers go)
    try:
        planned, plain = defn.compile(fun, x, 0.5, fuse=fuse), defn.compile(fun, x, 0.5)
        for rate in (0.5, 0.5, 0.5, 0.5, 2.0, 0.25, 0.5):
            for g, w in zip(planned(x, rate), plain._walk([x, Nx.to_tensor(rate)])):
                assert_bits_equal(g, w, f"rate {rate}")
        assert planned.replay is not None
    finally:
        Nx.default_backend(*previous)


def groups_and_operands(hip):
    rng = np.random.default_rng(17)
    key = Random.key(3, backend=hip)
    q, k = rand_float(rng, "bf16", (2, 40, 128), hip), rand_float(rng, "bf16", (2, 72, 128), hip)
    ragged = rand_float(rng, "f32", (37, 185), hip), rand_float(rng, "f32", (185,), hip)
    return {"words": (lambda kk: Random.normal(kk, shape=(1001,))[0], (key,)), "scores": (lambda a, b: attention_probabilities(a, b, 2), (q, k)),
            "ragged rows": (centred_and_scaled, ragged), "ragged sums": (lambda a, b: Nx.sum(Nx.exp(Nx.add(a, b)), axes=[1]), ragged)}


@pytest.mark.parametrize("met", ["inside the capture", "before the capture"])
@pytest.mark.parametrize("name", ["words", "scores", "ragged rows", "ragged sums"])
def test_groups_met_inside_a_capture(name, met, hip):
    """A group that a capture meets first is evaluated without its kernel there, one met before with it: every replay gives the bits
    of the evaluator, on new operands too, with work of its own between the replays.  (Scores on whole numbers: the kernel
    that contracts them adds in another order.)"""
    from nx_amd import backend as B
    fun, args = groups_and_operands(hip)[name]

    def fresh(i):
        out = []
        for t in args:
            v = np.roll(hip.to_numpy(t), i + 1, axis=0)
            if name == "scores":
                v = np.random.default_rng(i).integers(-2, 3, size=t.shape).astype(np.float32)
                v = (v.view(np.uint32) >> 16).astype(np.uint16)
            out.append(from_numpy(v + np.uint32(i) if name == "words" else v, t.type, hip))
        return out
    held = fresh(0)
    planned, plain = defn.compile(fun, *args, fuse="compiled"), defn.compile(fun, *args)
    if met == "before the capture":
        for _ in range(2):
            planned._walk(held)
    plain._walk(held)  # (the pool has the blocks that a capture takes)
    B.sync()
    B.capture_begin(0)
    try:
        results = planned._evaluate(held)
    finally:
        graph = B.capture_end(0)
    try:
        for i in (1, 2, 1, 3):
            now = fresh(i)
            for h, n in zip(held, now):
                B.copy_into(h, n)
            graph.launch()
            for g, w in zip(results, plain._walk(now)):
                assert_bits_equal(g, w, f"{name}, replay {i}")
            B.sync()
    finally:
        graph.destroy()


# K of one to eight steps of 32, whole and partial slabs of the contraction's own kernel; every form of the row, odd queries
@pytest.mark.parametrize("ty", ["bf16", "f16"])
@pytest.mark.parametrize("queries,keys,K", [(17, 64, 32), (16, 100, 96), (40, 300, 96), (33, 513, 64), (31, 1000, 160), (20, 1001, 256), (64, 776, 128), (1, 272, 64)])
def test_contracted_scores_are_rounded_sums(queries, keys, K, ty, hip):
    """The scores themselves, carried out of the kernel (halves, less nothing of their row's maximum).  Each is the operands' type's rounding (bf16 drops the
    low bits, f16 rounds to nearest: both rise with their argument) of an f32 sum of K exact products, which is at most K * 2^-24
    of the sum of their magnitudes away from the exact one: it lies between the roundings of the ends of that range."""
    rng = np.random.default_rng(seed_of(queries, keys, K, ty, "rounded"))
    heads = 2
    batch = 2 if keys * K <= 65536 else 128 // ((queries + 15) // 16)  # (over a large right operand: blocks for every CU)
    q, k = rand_float(rng, ty, (batch, queries, heads * K), hip), rand_float(rng, ty, (batch, keys, heads * K), hip)

    def fun(a, b):
        s = Nx.dot(split_heads(a, heads), [3], [0, 1], split_heads(b, heads), [3], [0, 1])
        half = Nx.multiply(Nx.as_type(s, "f32"), 0.5)
        return Nx.subtract(half, Nx.multiply(Nx.reduce_max(half, axes=[-1], keep_axes=True), 0.0))
    planned = defn.compile(fun, q, k, fuse="compiled")
    assert planned.roots[0].data.args[0].scores is not None
    calls, original = [], hip.fused_scores.__func__

    def counting(cls, *a, **kw):
        out = original(cls, *a, **kw)
        calls.append(1)
        return out
    hip.fused_scores = classmethod(counting)
    try:
        got = 2.0 * hip.to_numpy(planned(q, k)).astype(np.float64)
    finally:
        hip.fused_scores = classmethod(original)
    assert calls == [1]

    def heads_of(t):
        v = Nx.to_float64(t).reshape(t.shape[0], t.shape[1], heads, K)
        return v.transpose(0, 2, 1, 3)
    a, b = heads_of(q), heads_of(k).transpose(0, 1, 3, 2)
    exact, away = a @ b, K * 2.0 ** -24 * (np.abs(a) @ np.abs(b))

    def rounded(v):
        v = v.astype(np.float32)
        return (v.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32) if ty == "bf16" else v.astype(np.float16)
    lo, hi = rounded(exact - away).astype(np.float64), rounded(exact + away).astype(np.float64)
    assert (lo <= got).all() and (got <= hi).all(), (np.abs(got - exact).max(), int(((got < lo) | (got > hi)).sum()))
    # the range is 2 K 2^-24 * 0.64 K wide on these operands, at most two thirds of a unit of the results around sqrt(K) (f16, K = 256): a
    # quarter of them and more are decided to the bit, the others to a unit
    assert (lo == hi).mean() > 0.25
