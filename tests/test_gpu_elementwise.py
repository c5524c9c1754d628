"""Device element-wise ops and as_type against the CPU oracle on the same seeded inputs.

Bar: integer results bit-exact; f32/f16/bf16/f64 + - * / bit-exact (a correctly rounded op equals
the reference's f64-then-round); transcendental functions within 1e-5 relative (the tolerance the
target states for f32 element-wise ops) plus a denormal-sized absolute slack."""
import numpy as np
import pytest

from nx_amd import nx as Nx
from nx_amd import types as T
from support import _uint, assert_all_close, assert_bits_equal, from_numpy, raw, seed_of, values

pytestmark = pytest.mark.gpu

INT_TYPES = ["u8", "u16", "u32", "u64", "s8", "s16", "s32", "s64"]
FLOAT_TYPES = ["f16", "bf16", "f32", "f64"]
RTOL = 1e-5


def rand_raw(rng, ty, shape, lo=-4.0, hi=4.0, positive=False):
    """Random raw element array of Nx type `ty` (bf16 as uint16 bits); floats uniform in [lo, hi)."""
    ty = T.normalize(ty)
    if ty[0] in ("u", "s"):
        info = np.iinfo(T.numpy_dtype(ty))
        small = rng.integers(max(info.min, -100), min(info.max, 100) + 1, size=shape)
        wide = rng.integers(info.min, info.max, size=shape, dtype=T.numpy_dtype(ty), endpoint=True)
        pick = rng.random(shape) < 0.8
        return np.where(pick, small.astype(T.numpy_dtype(ty)), wide).astype(T.numpy_dtype(ty))
    x = rng.uniform(0.05 if positive else lo, hi, size=shape)
    if ty == ("bf", 16):
        return (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return x.astype(T.numpy_dtype(ty))


def both(arr, ty, hip, oracle):
    return from_numpy(arr, ty, hip), from_numpy(arr, ty, oracle)


EXACT_FLOAT = {"add", "subtract", "multiply", "divide", "min", "max", "equal", "not_equal", "greater", "less",
               "greater_equal", "less_equal", "logical_and", "logical_or", "logical_xor"}
ALL_BINARY = ["add", "subtract", "multiply", "divide", "pow", "remainder", "atan2", "min", "max", "equal",
              "not_equal", "greater", "less", "greater_equal", "less_equal", "logical_and", "logical_or",
              "logical_xor"]
INT_BINARY = ["quotient", "bitwise_and", "bitwise_or", "bitwise_xor", "left_shift", "right_shift"]


@pytest.mark.parametrize("op", ALL_BINARY)
@pytest.mark.parametrize("lt,rt", [("f32", "f32"), ("bf16", "bf16"), ("f16", "f16"), ("f64", "f64"), ("f32", "bf16"),
                                   ("s32", "f32"), ("u8", "f16"), ("f32", "f64"), ("s8", "bf16")])
def test_binary_float(op, lt, rt, hip, oracle):
    rng = np.random.default_rng(seed_of(op, lt, rt))
    shape = (37, 24)
    pos = op in ("pow",)
    a = rand_raw(rng, lt, shape, positive=pos)
    b = rand_raw(rng, rt, shape, positive=pos)
    if op in ("remainder", "divide") and T.is_integer(T.normalize(rt)):
        b = np.where(b == 0, 1, b).astype(b.dtype)
    if op == "pow":  # keep results inside f16 range
        a = rand_raw(rng, lt, shape, lo=0.5, hi=2.0) if T.is_float(T.normalize(lt)) else np.abs(a % 3).astype(a.dtype) + 1
        b = rand_raw(rng, rt, shape, lo=-2.0, hi=2.0) if T.is_float(T.normalize(rt)) else (b % 3).astype(b.dtype)
    if op == "multiply" and "f16" in (lt, rt):
        pass
    ha, oa = both(a, lt, hip, oracle)
    hb, ob = both(b, rt, hip, oracle)
    got, want = getattr(Nx, op)(ha, hb), getattr(Nx, op)(oa, ob)
    if op in EXACT_FLOAT:
        assert_bits_equal(got, want, f"{op} {lt} {rt}")
    else:
        assert_all_close(got, want, RTOL if got.type[1] >= 32 else 2.0 ** -7, 1e-30, f"{op} {lt} {rt}")


@pytest.mark.parametrize("op", ["add", "subtract", "multiply", "pow", "remainder", "min", "max", "equal", "not_equal",
                                "greater", "less", "greater_equal", "less_equal", "logical_and", "logical_xor"]
                         + INT_BINARY)
@pytest.mark.parametrize("lt,rt", [("s32", "s32"), ("u8", "u8"), ("s8", "u8"), ("s64", "s64"), ("u64", "u64"),
                                   ("u16", "s32"), ("s16", "s64"), ("u32", "u32"), ("u32", "s8")])
def test_binary_integer_is_bit_exact(op, lt, rt, hip, oracle):
    rng = np.random.default_rng(seed_of(op, lt, rt))
    shape = (5, 41)
    a, b = rand_raw(rng, lt, shape), rand_raw(rng, rt, shape)
    if op in ("remainder", "quotient"):
        b = np.where(b == 0, 1, b).astype(b.dtype)
    if op in ("left_shift", "right_shift"):
        b = (np.abs(b.astype(np.int64)) % 70).astype(b.dtype)
        b = np.where(b.astype(np.int64) < 0, 0, b).astype(b.dtype)
    if op == "pow":
        b = (np.abs(b.astype(np.int64)) % 6).astype(b.dtype)
        b = np.where(b.astype(np.int64) < 0, 0, b).astype(b.dtype)
    if lt == "u64" or rt == "u64":
        # u64 values >= 2^63 mixed with signed operands are a documented divergence; stay below
        a = (a >> 1).astype(a.dtype) if lt == "u64" else a
        b = (b >> 1).astype(b.dtype) if rt == "u64" else b
        if op in ("remainder", "quotient"):
            b = np.where(b == 0, 1, b).astype(b.dtype)
        if op in ("left_shift", "right_shift"):
            b = (b % 70).astype(b.dtype)
        if op == "pow":
            b = (b % 6).astype(b.dtype)
    ha, oa = both(a, lt, hip, oracle)
    hb, ob = both(b, rt, hip, oracle)
    assert_bits_equal(getattr(Nx, op)(ha, hb), getattr(Nx, op)(oa, ob), f"{op} {lt} {rt}")


BROADCASTS = [((64, 48), (64, 48)), ((64, 48), ()), ((), (64, 48)), ((64, 48), (48,)), ((48,), (64, 48)),
              ((4, 16, 24), (4, 16, 1)), ((4, 16, 1), (4, 16, 24)), ((3, 1, 5), (1, 7, 1)), ((2, 3, 4, 5), (3, 1, 5)),
              ((1,), (1,)), ((7, 13), (7, 1)), ((7, 13), (1, 13)), ((5, 3, 8), (3, 8)), ((9,), (6, 1)),
              ((2, 2, 2, 2, 2, 3), (2, 1, 2, 1, 2, 1)), ((1000003,), ())]


@pytest.mark.parametrize("ls,rs", BROADCASTS, ids=[f"{a}x{b}" for a, b in BROADCASTS])
@pytest.mark.parametrize("ty", ["f32", "bf16", "s32", "u8", "f64"])
def test_broadcasting_shapes(ls, rs, ty, hip, oracle):
    rng = np.random.default_rng(seed_of(ls, rs, ty))
    a, b = rand_raw(rng, ty, ls), rand_raw(rng, ty, rs)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    for op in ("add", "multiply", "greater"):
        assert_bits_equal(getattr(Nx, op)(ha, hb), getattr(Nx, op)(oa, ob), f"{op} {ls} {rs} {ty}")


@pytest.mark.parametrize("ty,shape", [("f32", (1016, 264)), ("bf16", (2040, 264)), ("s32", (1016, 264))])
def test_two_dense_operands_of_a_megabyte_take_two_vectors_per_lane(ty, shape, hip, oracle):
    """From 65536 vectors on, x + y of two dense tensors gives a lane two vectors, 256 apart: the last work-group
    here is partly filled, some of its lanes with a first vector and no second."""
    rng = np.random.default_rng(seed_of(ty, shape, "two vectors"))
    a, b = rand_raw(rng, ty, shape), rand_raw(rng, ty, shape)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    for op in ("add", "subtract", "multiply", "max", "less"):
        assert_bits_equal(getattr(Nx, op)(ha, hb), getattr(Nx, op)(oa, ob), f"{op} {ty} {shape}")


def test_scalar_number_operand(hip, oracle):
    rng = np.random.default_rng(5)
    a = rand_raw(rng, "f32", (33, 65))
    ha, oa = both(a, "f32", hip, oracle)
    for op, num in (("multiply", 0.5), ("add", 3), ("subtract", 1.25), ("divide", 8), ("max", 0.0), ("pow", 2)):
        assert_bits_equal(getattr(Nx, op)(ha, num), getattr(Nx, op)(oa, num), f"{op} tensor,{num}") if op != "pow" else \
            assert_all_close(getattr(Nx, op)(ha, num), getattr(Nx, op)(oa, num), RTOL, 0, "pow")
        if op not in ("pow",):
            assert_bits_equal(getattr(Nx, op)(num, ha), getattr(Nx, op)(num, oa), f"{op} {num},tensor")


MATH = ["exp", "expm1", "log", "log1p", "sigmoid", "cos", "sin", "tan", "cosh", "sinh", "tanh", "acos", "asin", "atan",
        "acosh", "asinh", "atanh", "sqrt", "rsqrt", "cbrt", "erf", "erfc", "erf_inv"]
DOMAIN = {"log": (0.01, 50), "log1p": (-0.9, 50), "acos": (-1, 1), "asin": (-1, 1), "acosh": (1.0, 50),
          "atanh": (-0.99, 0.99), "sqrt": (0, 50), "rsqrt": (0.01, 50), "erf_inv": (-0.99, 0.99), "exp": (-20, 10),
          "expm1": (-20, 10), "cosh": (-9, 9), "sinh": (-9, 9), "tan": (-1.5, 1.5)}


@pytest.mark.parametrize("op", MATH)
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16", "f64", "s32", "u8"])
def test_unary_math(op, ty, hip, oracle):
    rng = np.random.default_rng(seed_of(op, ty))
    lo, hi = DOMAIN.get(op, (-8, 8))
    if T.is_float(T.normalize(ty)):
        x = rand_raw(rng, ty, (4099,), lo=lo, hi=hi)
    else:
        x = rng.integers(max(int(np.ceil(lo)), 0 if ty == "u8" else -8), int(np.floor(hi)) + 1, size=(4099,)).astype(T.numpy_dtype(T.normalize(ty)))
        if op in ("atanh", "erf_inv"):
            x = np.zeros_like(x)
        if op in ("rsqrt", "log"):
            x = np.maximum(x, 1).astype(x.dtype)
    hx, ox = both(x, ty, hip, oracle)
    got, want = getattr(Nx, op)(hx), getattr(Nx, op)(ox)
    bits = got.type[1]
    # parity unpinned for erf_inv / cbrt / erf / erfc last bits: the reference delegates to the
    # `complex` package; libm-grade agreement is what is checked
    rtol = {16: 2.0 ** -7 if got.type[0] == "bf" else 2.0 ** -10, 32: RTOL, 64: 1e-12}[bits]
    if op in ("erf_inv",) and bits == 64:
        rtol = 1e-9
    assert_all_close(got, want, rtol, 1e-37 if bits == 32 else 1e-7 if bits == 16 else 1e-300, f"{op} {ty}")


@pytest.mark.parametrize("where", ["everywhere", "around the switch of polynomials", "next to one", "tiny", "powers of two from one"])
def test_f32_erf_inv_is_the_reference_but_for_last_bits_next_to_a_tie(where, hip, oracle):
    """The f32 kernel has its own logarithm and fuses the polynomials' steps: a few 1e-16 away from the reference's f64
    value, so a result can differ (by its last bit) only where that value is within 1e-15 of halfway between two floats,
    about one result in 2^25."""
    rng = np.random.default_rng(seed_of("erf_inv", where))
    x = {"everywhere": rng.uniform(-1, 1, 200_000), "around the switch of polynomials": rng.uniform(0.9965, 0.9968, 50_000),
         "next to one": 1 - np.arange(1, 5000) * 2.0 ** -24, "tiny": rng.uniform(-1, 1, 5000) * 10.0 ** rng.integers(-44, -3, 5000),
         "powers of two from one": 1 - 2.0 ** -np.arange(1, 25)}[where].astype(np.float32)
    got = values(Nx.erf_inv(from_numpy(x, "f32", hip))).astype(np.float32)
    want = values(Nx.erf_inv(from_numpy(x, "f32", oracle))).astype(np.float32)
    apart = np.abs(got.view(np.int32).astype(np.int64) - want.view(np.int32))
    assert apart.max() <= 1 and (apart != 0).sum() <= 2


def test_f32_erf_inv_rounds_its_nearest_misses_of_a_tie_as_the_exact_formula_does(hip):
    """Of the floats in [2^-10, 1) those whose value lies nearest to halfway between two floats, 3.9e-16 to 3.7e-15 of it away: the
    kernel's f64 value is within 2.9e-16 up to 0.9966, so each rounds as the formula in 80 bits does."""
    x = np.array([0x3C73BC07, 0x3BC4B808, 0x3F78AE99, 0x3C2A3771, 0x3B3C23F9], dtype=np.uint32).view(np.float32)
    x = np.concatenate([x, -x])
    wide = x.astype(np.longdouble)
    if np.finfo(np.longdouble).nmant < 63:
        pytest.skip("no 80-bit floats here")
    w = -np.log((1 - wide) * (1 + wide)) - np.longdouble(2.5)
    p = np.zeros_like(w)
    for c in (2.81022636e-08, 3.43273939e-07, -3.5233877e-06, -4.39150654e-06, 0.00021858087, -0.00125372503, -0.00417768164, 0.246640727, 1.50140941):
        p = p * w + np.longdouble(np.float64(c))
    got = values(Nx.erf_inv(from_numpy(x, "f32", hip))).astype(np.float32)
    assert np.array_equal(got.view(np.uint32), (p * wide).astype(np.float32).view(np.uint32))


@pytest.mark.parametrize("op", ["abs", "negate", "sign", "ceil", "floor", "round", "is_nan", "is_infinity"])
@pytest.mark.parametrize("ty", FLOAT_TYPES + ["s8", "s32", "s64", "u8", "u32"])
def test_unary_exact(op, ty, hip, oracle):
    rng = np.random.default_rng(seed_of(op, ty))
    x = rand_raw(rng, ty, (1031,), lo=-300, hi=300)
    if T.is_float(T.normalize(ty)):
        f = x.astype(np.float32) if ty != "bf16" else x
        # sprinkle halves, zeros and (where the reference defines them) non-finites
        if ty != "bf16":
            x[:6] = np.array([0.5, -0.5, 1.5, -1.5, 0.0, -0.0], dtype=x.dtype)
            if op in ("abs", "negate", "is_nan", "is_infinity", "sign"):
                x[6:9] = np.array([np.inf, -np.inf, np.nan], dtype=x.dtype)
    hx, ox = both(x, ty, hip, oracle)
    assert_bits_equal(getattr(Nx, op)(hx), getattr(Nx, op)(ox), f"{op} {ty}")


@pytest.mark.parametrize("op", ["bitwise_not", "population_count", "count_leading_zeros"])
@pytest.mark.parametrize("ty", INT_TYPES)
def test_unary_bit_ops(op, ty, hip, oracle):
    rng = np.random.default_rng(seed_of(op, ty))
    x = rand_raw(rng, ty, (777,))
    x[:3] = np.array([0, 1, np.iinfo(x.dtype).max], dtype=x.dtype)
    hx, ox = both(x, ty, hip, oracle)
    assert_bits_equal(getattr(Nx, op)(hx), getattr(Nx, op)(ox), f"{op} {ty}")


ALL_TYPES = INT_TYPES + FLOAT_TYPES


def encode(values64, ty):
    """float64 values -> raw element array of a float type (bf16 by truncation)."""
    ty = T.normalize(ty)
    with np.errstate(over="ignore"):
        if ty == ("bf", 16):
            return (values64.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        return values64.astype(T.numpy_dtype(ty))


@pytest.mark.parametrize("src", ALL_TYPES)
@pytest.mark.parametrize("dst", ALL_TYPES)
def test_as_type_every_pair_is_bit_exact(src, dst, hip, oracle):
    if src == dst:
        pytest.skip("as_type to the same type is a no-op in the front end")
    rng = np.random.default_rng(seed_of(src, dst))
    sty, dty = T.normalize(src), T.normalize(dst)
    f16_involved = ("f", 16) in (sty, dty)  # the reference raises when a finite value overflows f16
    if T.is_float(sty):
        lim = 60000.0 if f16_involved else 70000.0
        v = rng.uniform(-lim, lim, size=2053)
        special = [0.0, -0.0, 0.5, -0.5, 1e-3, 255.7, -255.7, 1e-7, 6.1e-5, np.inf, -np.inf, np.nan]
        if not f16_involved:  # wrap-around of float -> integer beyond 32 and 64 bits
            special += [3.0e9, -3.0e9, 1.0e19, -1.0e19, 5.0e18, 3.4e38]
        v[:len(special)] = special
        x = encode(v, src)
    else:
        x = rand_raw(rng, src, (2053,))
        if dty == ("f", 16):
            x = np.clip(x.astype(np.float64), -60000, 60000).astype(x.dtype)
    hx, ox = both(x, src, hip, oracle)
    assert_bits_equal(Nx.as_type(hx, dst), Nx.as_type(ox, dst), f"as_type {src}->{dst}")


def test_nan_is_written_canonically(hip, oracle):
    x = np.array([0x7FC00001, 0xFFC12345, 0x7F800001], dtype=np.uint32).view(np.float32)
    hx, ox = both(x, "f32", hip, oracle)
    for op in ("negate", "abs", "exp"):
        assert_bits_equal(getattr(Nx, op)(hx), getattr(Nx, op)(ox), op)
    assert_bits_equal(Nx.add(hx, 1.0), Nx.add(ox, 1.0), "add")
    assert_bits_equal(Nx.as_type(hx, "bf16"), Nx.as_type(ox, "bf16"), "as_type bf16")


DEEP = [((2, 3, 8, 16), (2, 1, 1, 16)), ((2, 3, 8, 16), (2, 1, 8, 1)), ((2, 3, 8, 16), (3, 1, 1)), ((2, 3, 8, 16), (1, 3, 1, 16)),
        ((4, 5, 24), (4, 1, 24)), ((4, 5, 24), (1, 5, 1)), ((3, 2, 4, 2, 16), (3, 1, 4, 1, 16)), ((2, 3, 8, 12), (2, 1, 1, 12)),
        ((6, 1, 7, 40), (1, 5, 1, 40)), ((2, 3, 5, 64), (2, 3, 1, 1))]


@pytest.mark.parametrize("ls,rs", DEEP, ids=[f"{a}-{b}" for a, b in DEEP])
@pytest.mark.parametrize("ty", ["f32", "bf16", "s32", "u8", "f64"])
@pytest.mark.parametrize("op", ["add", "multiply", "less", "max"])
def test_broadcasts_over_separated_axes(ls, rs, ty, op, hip, oracle):
    """A mask [b, 1, 1, s] against scores [b, h, s, s], a per-head scale [h, 1, 1], a per-row term [b, 1, s, 1]: the
    index space collapses to three or four axes, not to [rows, columns]; the vector kernel takes the row number
    apart.  Both operand orders; shapes off the 8-element grid and rank 5 take the general kernel.  Bit for bit."""
    rng = np.random.default_rng(seed_of(ls, rs, ty, op, "deep"))
    a, b = rand_raw(rng, ty, ls, lo=-5, hi=5), rand_raw(rng, ty, rs, lo=-5, hi=5)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    f = getattr(Nx, op)
    assert_bits_equal(f(ha, hb), f(oa, ob), f"{op} {ty} {ls} {rs}")
    assert_bits_equal(f(hb, ha), f(ob, oa), f"{op} {ty} {rs} {ls}")


RAGGED = [((301, c), (c,)) for c in (2, 3, 5, 7, 12, 17, 33, 100)] + [((301, c), (301, 1)) for c in (2, 3, 7, 33)] + \
         [((1, 13), (77, 1)), ((4, 25, 3), (3,)), ((9, 10, 5), (9, 10, 1)), ((2, 3), (3,))]


@pytest.mark.parametrize("ls,rs", RAGGED, ids=[f"{a}-{b}" for a, b in RAGGED])
@pytest.mark.parametrize("ty", ["f32", "bf16", "s32", "u8", "f64", "s64"])
@pytest.mark.parametrize("op", ["add", "multiply", "less", "max", "quotient"])
def test_rows_that_are_not_whole_vectors(ls, rs, ty, op, hip, oracle):
    """x[N, 3] * w[3], x[N, 5] + b[N, 1], a column against a row: rows whose length is not a whole number of vectors are
    cut into vectors of the flat output (vectors run across row ends, the last one is partial).  Both operand orders,
    bit for bit; an integer quotient by non-zero divisors reports nothing for the lanes beyond the end."""
    rng = np.random.default_rng(seed_of(ls, rs, ty, op, "ragged"))
    a, b = rand_raw(rng, ty, ls, lo=1, hi=9), rand_raw(rng, ty, rs, lo=1, hi=9)
    if op == "quotient":
        if ty in ("f32", "bf16", "f64"):
            pytest.skip("quotient is an integer operation")
        a, b = np.where(a == 0, 1, a).astype(a.dtype), np.where(b == 0, 1, b).astype(b.dtype)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    f = getattr(Nx, op)
    assert_bits_equal(f(ha, hb), f(oa, ob), f"{op} {ty} {ls} {rs}")
    assert_bits_equal(f(hb, ha), f(ob, oa), f"{op} {ty} {rs} {ls}")
    from nx_amd import backend as B
    B.sync()  # nothing was recorded for a later wait to raise


DEEP_RAGGED = [((2, 3, 197, 197), (2, 1, 1, 197)), ((2, 3, 77, 77), (1, 3, 1, 1)), ((4, 7, 13), (4, 1, 13)), ((5, 9, 3), (1, 9, 1)),
               ((3, 5, 7, 11), (3, 1, 7, 1)), ((2, 4, 6, 9), (1, 4, 1, 9))]


@pytest.mark.parametrize("ls,rs", DEEP_RAGGED, ids=[f"{a}-{b}" for a, b in DEEP_RAGGED])
@pytest.mark.parametrize("ty", ["f32", "bf16", "s32", "u8"])
@pytest.mark.parametrize("op", ["add", "multiply", "less", "quotient"])
def test_broadcasts_over_separated_axes_off_the_vector_grid(ls, rs, ty, op, hip, oracle):
    """A mask [b, 1, 1, 197] against scores [b, h, 197, 197]: three or four collapsed axes AND rows that are not whole
    vectors -- vectors of the flat output, the row's operand offsets taken apart again where a row ends."""
    rng = np.random.default_rng(seed_of(ls, rs, ty, op, "deep ragged"))
    a, b = rand_raw(rng, ty, ls, lo=1, hi=9), rand_raw(rng, ty, rs, lo=1, hi=9)
    if op == "quotient":
        if ty in ("f32", "bf16"):
            pytest.skip("quotient is an integer operation")
        a, b = np.where(a == 0, 1, a).astype(a.dtype), np.where(b == 0, 1, b).astype(b.dtype)
    if int(np.prod(ls)) > 60000:  # the oracle's loops: a corner of the big case, numpy for the rest
        got = hip.to_numpy(getattr(Nx, op)(from_numpy(a, ty, hip), from_numpy(b, ty, hip)))
        sub = (slice(0, 1), slice(0, 2), slice(0, 50), slice(None))
        bs = tuple(s_ if d != 1 else slice(None) for s_, d in zip(sub, rs))
        want = getattr(Nx, op)(from_numpy(np.ascontiguousarray(a[sub]), ty, oracle), from_numpy(np.ascontiguousarray(b[bs]), ty, oracle))
        assert np.array_equal(np.ascontiguousarray(got[sub]).view(np.uint8), oracle.to_numpy(want).view(np.uint8) if hasattr(oracle, "to_numpy") else np.frombuffer(Nx.to_binary(want), dtype=np.uint8).reshape(np.ascontiguousarray(got[sub]).view(np.uint8).shape))
        if op in ("add", "multiply") and ty in ("f32", "s32"):
            assert np.array_equal(got, (a + b) if op == "add" else (a * b))
        return
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    f = getattr(Nx, op)
    assert_bits_equal(f(ha, hb), f(oa, ob), f"{op} {ty} {ls} {rs}")
    assert_bits_equal(f(hb, ha), f(ob, oa), f"{op} {ty} {rs} {ls}")


@pytest.mark.parametrize("ty", ["f16", "bf16", "f32", "f64"])
@pytest.mark.parametrize("op", ["multiply", "divide", "add", "subtract"])
@pytest.mark.parametrize("form", ["same_shape", "one_per_row", "one_row", "a_number"])
def test_signed_zeros_through_every_operand_form(ty, op, form, hip, oracle):
    """The sign of a zero result: (-x) * 0 = -0, 0 / (-x) = -0, -0 + -0 = -0, x - x = +0, in the kernels for operands of
    one shape and in those that spread one operand along or across the rows (a product followed by the rounding to f16
    once came out of the compiler as one instruction that added +0 to it)."""
    rng = np.random.default_rng(seed_of("signed zeros", ty, op, form))
    dtype = np.float32 if ty == "bf16" else T.numpy_dtype(T.normalize(ty))
    shape = {"same_shape": (64, 256), "one_per_row": (64, 1), "one_row": (256,), "a_number": ()}[form]
    a = rng.choice(np.array([0.0, -0.0, 1.25, -1.25, 3.0, -0.5], dtype), size=(64, 256))
    b = rng.choice(np.array([0.0, -0.0, 2.0, -2.0], dtype), size=shape)
    if ty == "bf16":
        a, b = [(np.asarray(v, np.float32).view(np.uint32) >> 16).astype(np.uint16) for v in (a, b)]
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    for flip in (False, True):  # (a float divided by zero is an infinity or a NaN in the reference, not an error)
        got = getattr(Nx, op)(hb, ha) if flip else getattr(Nx, op)(ha, hb)
        want = getattr(Nx, op)(ob, oa) if flip else getattr(Nx, op)(oa, ob)
        assert_bits_equal(got, want, f"{op} {ty} {form} flipped={flip}")


MATH = ["exp", "expm1", "log", "log1p", "sigmoid", "cos", "sin", "tan", "cosh", "sinh", "tanh", "acos", "asin", "atan", "acosh",
        "asinh", "atanh", "sqrt", "rsqrt", "cbrt", "erf", "erfc", "erf_inv", "abs", "negate", "floor", "ceil", "round", "sign"]


@pytest.mark.parametrize("ty", ["f16", "bf16", "f32", "f64"])
@pytest.mark.parametrize("op", MATH)
def test_unary_results_that_are_zero_or_not_finite_have_the_reference_bits(op, ty, hip, oracle):
    """Zeros of either sign, the smallest numbers, ones, the ends of the domains, infinities and NaN: wherever the
    reference's result is a zero, an infinity or NaN the device's is the same bits (sin(-0) = -0, tanh of a tiny negative
    number that rounds to zero keeps its sign, log(0) = -inf, ...); elsewhere the tolerance of the other tests applies."""
    tiny = {"f16": 6e-8, "bf16": 1e-38, "f32": 1e-45, "f64": 5e-324}[ty]
    from oracle.binary_backend import ReferenceRaises
    large = 8.0 if ty == "f16" else 30.0  # (a finite result beyond f16's range raises in the reference)
    v = np.array([0.0, -0.0, tiny, -tiny, 1.0, -1.0, 0.5, -0.5, 2.0, -2.0, np.inf, -np.inf, np.nan, 1e-4, -1e-4, large, -large])
    x = encode(v, ty)
    hx, ox = both(x, ty, hip, oracle)
    try:
        want = getattr(Nx, op)(ox)
    except ReferenceRaises as e:
        pytest.skip(f"the reference raises: {e}")
    got = getattr(Nx, op)(hx)
    assert got.type == want.type and got.shape == want.shape
    g, w = raw(got), raw(want)
    gf, wf = values(got), values(want)
    fixed = (wf == 0) | ~np.isfinite(wf)
    gb, wb = g.view(_uint(g.dtype)), w.view(_uint(w.dtype))
    assert np.array_equal(gb[fixed], wb[fixed]), f"{op} {ty}: inputs {v[fixed][gb[fixed] != wb[fixed]]} got {gf[fixed][gb[fixed] != wb[fixed]]} want {wf[fixed][gb[fixed] != wb[fixed]]}"
    rest = ~fixed
    tol = {"f16": 2e-3, "bf16": 1.6e-2, "f32": 2e-6, "f64": 1e-12}[ty]
    assert np.all(np.abs(gf[rest] - wf[rest]) <= tol * np.abs(wf[rest])), f"{op} {ty}: {gf[rest]} vs {wf[rest]}"


@pytest.mark.parametrize("ty", ["f16", "bf16", "f32", "f64"])
@pytest.mark.parametrize("op", ["add", "subtract", "multiply", "divide", "pow", "atan2", "min", "max", "remainder"])
def test_binary_results_that_are_zero_or_not_finite_have_the_reference_bits(op, ty, hip, oracle):
    """Every pair from zeros of either sign, the smallest numbers, small integers (odd and even), a half, infinities and
    NaN (the special cases of pow, atan2 and division among them), as operands of one shape and with a number on either
    side; results that are a zero, an infinity or NaN must be the reference's bits."""
    from oracle.binary_backend import ReferenceRaises
    tiny = {"f16": 6e-8, "bf16": 1e-38, "f32": 1e-45, "f64": 5e-324}[ty]
    s = np.array([0.0, -0.0, tiny, -tiny, 1.0, -1.0, 2.0, -2.0, 3.0, -3.0, 0.5, -0.5, np.inf, -np.inf, np.nan])
    if op == "remainder":  # :math.fmod raises for a zero divisor and for operands that are not finite
        s = s[np.isfinite(s) & (s != 0)]
    a, b = [g.ravel() for g in np.meshgrid(s, s, indexing="ij")]
    if op in ("divide", "pow") and ty != "f64":  # a finite result beyond the type's range raises in the reference: not asked
        with np.errstate(all="ignore"):
            exact = np.divide(a, b) if op == "divide" else np.power(a, b)
        fits = ~(np.isfinite(exact) & (np.abs(exact) > (65504.0 if ty == "f16" else 3.4e38)))
        a, b = a[fits], b[fits]
    ha, oa = both(encode(a, ty), ty, hip, oracle)
    hb, ob = both(encode(b, ty), ty, hip, oracle)
    try:
        want = getattr(Nx, op)(oa, ob)
    except ReferenceRaises as e:
        pytest.skip(f"the reference raises: {e}")
    got = getattr(Nx, op)(ha, hb)
    g, w = raw(got), raw(want)
    gf, wf = values(got), values(want)
    fixed = (wf == 0) | ~np.isfinite(wf)
    gb, wb = g.view(_uint(g.dtype)), w.view(_uint(w.dtype))
    bad = fixed & (gb != wb)
    assert not bad.any(), f"{op} {ty}: a {a[bad]} b {b[bad]} got {gf[bad]} want {wf[bad]}"
    rest = ~fixed
    tol = {"f16": 2e-3, "bf16": 1.6e-2, "f32": 2e-6, "f64": 1e-12}[ty]
    assert np.all(np.abs(gf[rest] - wf[rest]) <= tol * np.abs(wf[rest])), f"{op} {ty}"


@pytest.mark.parametrize("lt", ["s8", "u8", "s16", "u16", "s32", "u32", "s64", "u64"])
@pytest.mark.parametrize("rt", ["s8", "u8", "s32", "u32", "s64", "u64"])
@pytest.mark.parametrize("op", ["add", "subtract", "multiply", "quotient", "remainder", "min", "max", "less", "equal",
                                "bitwise_and", "bitwise_or", "bitwise_xor", "left_shift", "right_shift"])
def test_integer_extremes_in_every_pair_of_types(op, lt, rt, hip, oracle):
    """Every pair from the ends of each type, the values next to them, zero, one and minus one: the most negative number
    divided by -1, products and sums that wrap, an unsigned operand beyond the signed range against a negative one, shift
    counts up to the width and beyond (negative counts and zero divisors raise in the reference: left out)."""
    order_matters = ("quotient", "remainder", "min", "max", "less", "equal", "right_shift")
    if op in order_matters and "u64" in (lt, rt) and "s" in (lt[0], rt[0]):
        # known difference: a u64 operand against a signed one is computed in the s64 class, where values of 2^63 and more
        # read as negative; the reference keeps them positive (unbounded integers).  Sums, products and bitwise results
        # wrap to the same bits either way and are checked below.
        pytest.skip("u64 values of 2^63 and more against a signed operand: compared, divided and shifted as negative s64")

    def ends(ty):
        info = np.iinfo(T.numpy_dtype(T.normalize(ty)))
        vals = {info.min, info.min + 1, info.max, info.max - 1, 0, 1, 2, 7}
        if info.min < 0:
            vals |= {-1, -2, -7}
        return np.array(sorted(vals), dtype=T.numpy_dtype(T.normalize(ty)))
    a, b = ends(lt), ends(rt)
    if op in ("quotient", "remainder"):
        b = b[b != 0]
    if op in ("left_shift", "right_shift"):
        b = np.array([0, 1, 7, 8, 31, 32, 63, 64, 65], dtype=np.int64).astype(b.dtype)
        b = np.unique(b[b >= 0])
    a, b = [g.ravel() for g in np.meshgrid(a, b, indexing="ij")]
    ha, oa = both(a, lt, hip, oracle)
    hb, ob = both(b, rt, hip, oracle)
    assert_bits_equal(getattr(Nx, op)(ha, hb), getattr(Nx, op)(oa, ob), f"{op} {lt} {rt}")


# A dense tensor with a row of its columns or with one value per row, where rows are not whole vectors of eight: fewer columns
# than a lane's vector, rows that are whole vectors of four, a last vector cut off; either operand the dense one.
@pytest.mark.parametrize("rows,cols", [(5, 2), (1001, 3), (77, 7), (33, 10), (513, 100), (1000, 33), (3, 1001), (129, 257), (2, 5)])
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("op", ["add", "subtract", "divide", "max", "atan2"])
def test_short_rows_with_a_row_or_a_value_per_row(rows, cols, ty, op, hip, oracle):
    rng = np.random.default_rng(seed_of("flat", rows, cols, ty, op))
    x = rand_raw(rng, ty, (rows, cols), lo=-4, hi=4)
    hx, ox = both(x, ty, hip, oracle)
    for shape in ((1, cols), (rows, 1)):
        y = rand_raw(rng, ty, shape, lo=1, hi=4)
        hy, oy = both(y, ty, hip, oracle)
        for (a, b), (c, d) in (((hx, hy), (ox, oy)), ((hy, hx), (oy, ox))):
            got, want = getattr(Nx, op)(a, b), getattr(Nx, op)(c, d)
            if op == "atan2":  # a library function on either side
                assert_all_close(got, want, {"f32": 1e-6, "bf16": 2.0 ** -7, "f16": 2.0 ** -10}[ty], 0, f"{op} {ty} {rows}x{cols} {shape}")
            else:
                assert_bits_equal(got, want, f"{op} {ty} {rows}x{cols} {shape}")


@pytest.mark.parametrize("rows,cols", [(40, 15), (33, 3), (9, 20), (1001, 2)])
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("op", ["add", "subtract", "multiply", "divide", "max", "min", "atan2"])
def test_short_rows_on_special_values(rows, cols, ty, op, hip, oracle):
    """Zeros of either sign, infinities and NaN on either side of a row or a value per row: the reference's bits wherever its
    result is a zero or not finite."""
    rng = np.random.default_rng(seed_of("flat special", rows, cols, ty, op))
    s = np.array([0.0, -0.0, 1.0, -1.0, 2.0, -3.0, 0.5, np.inf, -np.inf, np.nan])
    x = rng.choice(s, size=(rows, cols))
    hx, ox = both(encode(x, ty), ty, hip, oracle)
    for shape in ((1, cols), (rows, 1)):
        hy, oy = both(encode(rng.choice(s, size=shape), ty), ty, hip, oracle)
        for (a, b), (c, d) in (((hx, hy), (ox, oy)), ((hy, hx), (oy, ox))):
            got, want = getattr(Nx, op)(a, b), getattr(Nx, op)(c, d)
            g, w, gf, wf = raw(got), raw(want), values(got), values(want)
            fixed = (wf == 0) | ~np.isfinite(wf)
            assert np.array_equal(g.view(_uint(g.dtype))[fixed], w.view(_uint(w.dtype))[fixed]), f"{op} {ty} {rows}x{cols} {shape}"
            tol = {"f16": 2e-3, "bf16": 1.6e-2, "f32": 2e-6}[ty] if op == "atan2" else 0.0  # (a library function on either side)
            assert (np.abs(gf[~fixed] - wf[~fixed]) <= tol * np.abs(wf[~fixed])).all(), f"{op} {ty} {rows}x{cols} {shape}"


SPECIAL = [0.0, -0.0, 1.0, -1.5, np.inf, -np.inf, np.nan, 1e-40, -1e36, 6e-8, 60000.0]


# a whole number that counts, behind sums: one element, a wave, blocks and one element more, the longest the small kernel takes and one more
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("n", [1, 7, 256, 257, 65536, 65537])
@pytest.mark.parametrize("count", [1, 3, -7, 0, 20000, 16777217, -2147483648])
def test_quotients_by_a_whole_number(ty, n, count, hip, oracle):
    rng = np.random.default_rng(seed_of(ty, n, count, "count"))
    x = np.resize(np.concatenate([SPECIAL if ty != "f16" else [v for v in SPECIAL if abs(v) < 1e30 or not np.isfinite(v)], rng.uniform(-1e4, 1e4, size=256)]), n).astype(np.float32)
    arr = (x.view(np.uint32) >> 16).astype(np.uint16) if ty == "bf16" else x.astype(np.float16 if ty == "f16" else np.float32)
    h, o = both(arr, ty, hip, oracle)
    hc, oc = both(np.array(count, np.int32), "s32", hip, oracle)
    assert_bits_equal(Nx.divide(h, hc), Nx.divide(o, oc), f"{ty} [{n}] / {count}")


@pytest.mark.parametrize("shape", [(1,), (3,), (1024,), (1025,), (333, 250), (4, 5, 7)])
def test_values_times_a_mask(shape, hip, oracle):
    rng = np.random.default_rng(seed_of(shape, "mask"))
    x = np.resize(np.concatenate([SPECIAL, rng.uniform(-1e4, 1e4, size=500)]), shape).astype(np.float32)
    m = rng.choice(np.array([0, 1, 1, 255], np.uint8), size=shape)
    (hx, ox), (hm, om) = both(x, "f32", hip, oracle), both(m, "u8", hip, oracle)
    assert_bits_equal(Nx.multiply(hx, hm), Nx.multiply(ox, om), "x * mask")
    assert_bits_equal(Nx.multiply(hm, hx), Nx.multiply(om, ox), "mask * x")
