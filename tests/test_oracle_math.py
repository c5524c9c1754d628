"""Pins the oracle's 23 unary math functions and `atan2` / `pow` / `divide` / `remainder` by what the
mathematics fixes -- the reference holds almost no literal for them (its doctests print what the
function under test returns).

* every function against an arbitrary-precision evaluation (mpmath, 40 digits) on a grid over its
  domain: f64 results within 4 ulp, and f32 results -- computed in f64 and rounded once, as the
  reference does (`shared.ex:123-194`) -- equal to the correctly rounded f32 of the true value;
* the inverse pairs, the identities and the parities that relate the functions to each other;
* exact special values, and IEEE 754 / C Annex F results at zeros, infinities and NaN where the
  reference's arithmetic reduces to the C library (`:math.*` behind `Complex.*`).

A swapped pair (sin / cos, sinh / asinh, log / log1p), a dropped term (`exp(x) - 1`, `log(x + 1)`), a
wrong sign or a transposed `atan2` operand fails at least one of these."""
import math
import re
from pathlib import Path

import mpmath as mp
import numpy as np
import pytest

from nx_amd import nx as Nx
from support import from_numpy, raw, values

mp.mp.dps = 40


def run(name, x, ty, oracle):
    return getattr(Nx, name)(from_numpy(np.asarray(x, dtype=np.float64 if ty == "f64" else np.float32), ty, oracle))


def grid(lo, hi, n=41, log=False):
    if log:
        return np.exp(np.linspace(math.log(lo), math.log(hi), n))
    return np.linspace(lo, hi, n)


# name -> (arbitrary-precision function, points inside the domain)
SIGNED = np.concatenate([-grid(1e-3, 20, 25, log=True), grid(1e-3, 20, 25, log=True)])
POSITIVE = grid(1e-6, 1e6, 49, log=True)
UNIT = np.concatenate([grid(-0.999, 0.999, 41), [1e-9, -1e-9]])
FUNS = {
    "exp": (mp.exp, SIGNED), "expm1": (mp.expm1, SIGNED[np.abs(SIGNED) > 0.5]),  # exp(x) - 1 cancels near 0: its own test below
    "log": (mp.log, POSITIVE), "log1p": (mp.log1p, POSITIVE[POSITIVE > 0.5]),  # log(x + 1): same remark
    "sigmoid": (lambda x: 1 / (1 + mp.exp(-x)), SIGNED),
    "cos": (mp.cos, SIGNED), "sin": (mp.sin, SIGNED), "tan": (mp.tan, SIGNED),
    "cosh": (mp.cosh, SIGNED), "sinh": (mp.sinh, SIGNED), "tanh": (mp.tanh, SIGNED),
    "acos": (mp.acos, UNIT), "asin": (mp.asin, UNIT), "atan": (mp.atan, SIGNED),
    "acosh": (mp.acosh, 1 + POSITIVE), "asinh": (mp.asinh, SIGNED), "atanh": (mp.atanh, UNIT),
    "sqrt": (mp.sqrt, POSITIVE), "rsqrt": (lambda x: 1 / mp.sqrt(x), POSITIVE), "cbrt": (mp.cbrt, POSITIVE),
    "erf": (mp.erf, SIGNED[np.abs(SIGNED) < 6]), "erfc": (mp.erfc, SIGNED[np.abs(SIGNED) < 6]),
}


def ulp64(v):
    return np.spacing(np.abs(v))


@pytest.mark.parametrize("name", sorted(FUNS))
def test_f64_within_4_ulp_of_the_true_value(name, oracle):
    f, xs = FUNS[name]
    got = values(run(name, xs, "f64", oracle))
    want = np.array([float(f(mp.mpf(float(x)))) for x in xs])
    err = np.abs(got - want) / ulp64(want)
    assert err.max() <= 4, f"{name}: {err.max():.1f} ulp at x = {xs[int(err.argmax())]!r}"


@pytest.mark.parametrize("name", sorted(FUNS))
def test_f32_is_the_correctly_rounded_true_value(name, oracle):
    f, xs = FUNS[name]
    xs = xs.astype(np.float32)
    got = raw(run(name, xs, "f32", oracle))
    want = np.array([float(f(mp.mpf(float(x)))) for x in xs]).astype(np.float32)
    # computed in f64 and rounded once: only a true value within 2^-29 of a rounding boundary could differ
    assert (got.view(np.uint32) == want.view(np.uint32)).mean() >= 0.97, name
    assert np.abs(got.astype(np.float64) - want.astype(np.float64)).max() <= np.spacing(np.abs(want)).max()


def test_expm1_and_log1p_follow_the_reference_formulas_not_the_accurate_routines(oracle):
    # `exp(x) - 1` and `log(x + 1)` (shared.ex:314-330): the cancellation near 0 is part of the reference result
    x = np.array([1e-10, -1e-10, 1e-17, 3e-9])
    assert np.array_equal(values(run("expm1", x, "f64", oracle)), np.exp(x) - 1)
    assert np.array_equal(values(run("log1p", x, "f64", oracle)), np.log(x + 1))
    assert values(run("expm1", [1e-17], "f64", oracle)).item() == 0.0 and math.expm1(1e-17) != 0.0


def test_erf_inv_inverts_erf_and_follows_giles_polynomial_accuracy(oracle):
    # the reference's erf_inv is a single-precision polynomial evaluated in doubles: it inverts erf to ~1e-7,
    # not to double precision (its bit pattern is pinned by the transcribed Nx.Random.normal answers)
    p = np.linspace(-0.99, 0.99, 67)
    back = values(run("erf", values(run("erf_inv", p, "f64", oracle)), "f64", oracle))
    assert np.abs(back - p).max() < 5e-7
    true = np.array([float(mp.erfinv(mp.mpf(float(v)))) for v in p])
    got = values(run("erf_inv", p, "f64", oracle))
    assert np.abs(got - true).max() < 2e-6 and np.array_equal(np.sign(got), np.sign(p))
    assert values(run("erf_inv", [0.0], "f64", oracle)).item() == 0.0


def test_the_logarithm_of_the_f32_erf_inv_kernel_has_a_constant_to_2_57():
    """Its -2.5 - log c stands in one double that cancels e ln 2 next to zero: c is chosen for it (1/sqrt(2) misses by 2^-53)."""
    source = (Path(__file__).resolve().parent.parent / "nx_amd" / "csrc" / "elementwise_ops.cuh").read_text()
    body = source[source.index("float erf_inv_f32("):]
    c = float.fromhex(re.search(r"const double c = (\S+?),", body).group(1))
    constant = float.fromhex(re.search(r"fma_consts\(e, -0x1.62e42fefa39efp-1, (\S+?)\)", body).group(1))
    assert abs(c - 2 ** -0.5) < 1e-12
    with mp.workdps(50):
        assert abs(mp.mpf(constant) + mp.mpf(2.5) + mp.log(mp.mpf(c))) < mp.mpf(2) ** -57


INVERSE_PAIRS = [("acos", "cos", grid(0.01, 3.1, 31)), ("asin", "sin", grid(-1.5, 1.5, 31)), ("atan", "tan", grid(-1.5, 1.5, 31)),
                 ("acosh", "cosh", grid(0.1, 10, 31)), ("asinh", "sinh", grid(-10, 10, 31)), ("atanh", "tanh", grid(-3, 3, 31)),
                 ("log", "exp", grid(-20, 20, 31)), ("exp", "log", POSITIVE), ("sqrt", None, POSITIVE), ("cbrt", None, POSITIVE)]


@pytest.mark.parametrize("outer,inner,xs", INVERSE_PAIRS, ids=[f"{a}-{b}" for a, b, _ in INVERSE_PAIRS])
def test_inverse_pairs(outer, inner, xs, oracle):
    if inner is None:  # sqrt(x)^2 = x, cbrt(x)^3 = x
        r = values(run(outer, xs, "f64", oracle))
        back = r * r if outer == "sqrt" else r * r * r
    else:
        back = values(run(outer, values(run(inner, xs, "f64", oracle)), "f64", oracle))
    # the conditioning of the round trip is at most ~|x| / |f'(x)| ...: 1e-12 relative holds on these grids
    # except where the inner function flattens (acos near 0, atanh(tanh) at |x| = 3, acosh(cosh) at 0.1)
    loose = {"acos": 1e-9, "atanh": 1e-9, "acosh": 1e-9}.get(outer, 1e-12)
    assert np.allclose(back, xs, rtol=loose, atol=loose), f"{outer}({inner}(x)) != x: {np.abs(back - xs).max():.2e}"


def test_identities_between_the_functions(oracle):
    x = grid(-6, 6, 61)
    v = lambda n, a=x: values(run(n, a, "f64", oracle))  # noqa: E731
    close = lambda a, b: np.allclose(a, b, rtol=1e-12, atol=1e-12)  # noqa: E731
    assert close(v("sin") ** 2 + v("cos") ** 2, 1.0)
    assert close(v("cosh") ** 2 - v("sinh") ** 2, np.ones_like(x)) or np.allclose(v("cosh") ** 2 - v("sinh") ** 2, 1.0, rtol=0, atol=1e-9)
    assert close(v("tan"), v("sin") / v("cos"))
    assert close(v("tanh"), v("sinh") / v("cosh"))
    assert close(v("erf") + v("erfc"), 1.0)
    assert close(v("sigmoid") + v("sigmoid", -x), 1.0)
    assert close(v("exp") * v("exp", -x), 1.0)
    assert close(v("cosh"), (v("exp") + v("exp", -x)) / 2)
    assert close(v("sinh"), (v("exp") - v("exp", -x)) / 2)
    pos = POSITIVE
    assert close(v("rsqrt", pos) * v("sqrt", pos), 1.0)
    assert close(v("log", pos * pos), 2 * v("log", pos))
    # parities: odd / even functions keep exact symmetry
    for odd in ("sin", "tan", "sinh", "tanh", "asinh", "atan", "erf"):
        assert np.array_equal(v(odd, -x), -v(odd)), odd
    for odd in ("asin", "atanh"):
        assert np.array_equal(v(odd, -UNIT), -v(odd, UNIT)), odd
    for even in ("cos", "cosh"):
        assert np.array_equal(v(even, -x), v(even)), even
    assert close(v("acos", UNIT) + v("asin", UNIT), math.pi / 2)
    assert close(v("cbrt", pos), np.cbrt(pos)) and close(v("cbrt", np.array([27.0, 1e-3, 8.0])), [3.0, 0.1, 2.0])


EXACT = [("exp", 0.0, 1.0), ("expm1", 0.0, 0.0), ("log", 1.0, 0.0), ("log1p", 0.0, 0.0), ("sigmoid", 0.0, 0.5),
         ("cos", 0.0, 1.0), ("sin", 0.0, 0.0), ("tan", 0.0, 0.0), ("cosh", 0.0, 1.0), ("sinh", 0.0, 0.0), ("tanh", 0.0, 0.0),
         ("acos", 1.0, 0.0), ("asin", 0.0, 0.0), ("atan", 0.0, 0.0), ("acosh", 1.0, 0.0), ("asinh", 0.0, 0.0), ("atanh", 0.0, 0.0),
         ("sqrt", 4.0, 2.0), ("sqrt", 0.0, 0.0), ("rsqrt", 4.0, 0.5), ("cbrt", 8.0, 2.0), ("cbrt", 0.0, 0.0),
         ("erf", 0.0, 0.0), ("erfc", 0.0, 1.0), ("asin", 1.0, math.pi / 2), ("acos", -1.0, math.pi), ("atan", 1.0, math.pi / 4),
         ("exp", 1.0, math.e), ("log", math.e, 1.0)]


@pytest.mark.parametrize("name,x,want", EXACT, ids=[f"{n}({x})" for n, x, _ in EXACT])
def test_exact_special_values(name, x, want, oracle):
    got = values(run(name, [x], "f64", oracle)).item()
    assert got == want or abs(got - want) <= np.spacing(want), f"{name}({x}) = {got!r}, expected {want!r}"


# IEEE 754 limits the reference inherits from the C library for infinite and NaN arguments
NONFINITE = [("exp", math.inf, math.inf), ("exp", -math.inf, 0.0), ("expm1", -math.inf, -1.0), ("log", math.inf, math.inf),
             ("sigmoid", math.inf, 1.0), ("sigmoid", -math.inf, 0.0), ("tanh", math.inf, 1.0), ("tanh", -math.inf, -1.0),
             ("atan", math.inf, math.pi / 2), ("atan", -math.inf, -math.pi / 2), ("sqrt", math.inf, math.inf),
             ("rsqrt", math.inf, 0.0), ("cosh", -math.inf, math.inf), ("sinh", -math.inf, -math.inf), ("erf", math.inf, 1.0),
             ("erf", -math.inf, -1.0), ("erfc", math.inf, 0.0), ("erfc", -math.inf, 2.0), ("asinh", -math.inf, -math.inf),
             ("acosh", math.inf, math.inf), ("cbrt", math.inf, math.inf)]


@pytest.mark.parametrize("name,x,want", NONFINITE, ids=[f"{n}({x})" for n, x, _ in NONFINITE])
def test_limits_at_infinity(name, x, want, oracle):
    for ty in ("f64", "f32"):
        got = values(run(name, [x], ty, oracle)).item()
        assert got == want or abs(got - want) <= np.spacing(np.float32(abs(want))), f"{name}({x}) [{ty}] = {got!r}"


@pytest.mark.parametrize("name", sorted(FUNS) + ["erf_inv"])
def test_nan_in_nan_out(name, oracle):
    assert math.isnan(values(run(name, [math.nan], "f64", oracle)).item())
    bits = raw(run(name, [math.nan], "f32", oracle)).view(np.uint32).item()
    assert bits == 0x7FC00000, f"{name}: NaN is written with the canonical pattern (type.ex:128-158), got {bits:#x}"


def bin_op(name, a, b, ty, oracle):
    dt = np.float64 if ty == "f64" else np.float32
    return values(getattr(Nx, name)(from_numpy(np.asarray(a, dtype=dt), ty, oracle), from_numpy(np.asarray(b, dtype=dt), ty, oracle)))


def test_atan2_quadrants_and_axes(oracle):
    ys = np.array([1.0, 1.0, -1.0, -1.0, 0.0, 1.0, 0.0, -1.0, 3.0, -2.0])
    xs = np.array([1.0, -1.0, -1.0, 1.0, 1.0, 0.0, -1.0, 0.0, 4.0, 5.0])
    got = bin_op("atan2", ys, xs, "f64", oracle)
    want = np.array([float(mp.atan2(mp.mpf(float(y)), mp.mpf(float(x)))) for y, x in zip(ys, xs)])
    assert np.abs(got - want).max() <= 4e-16
    # the operand order: atan2(y, x), not atan2(x, y)
    assert bin_op("atan2", [1.0], [0.0], "f64", oracle).item() == math.pi / 2
    # C Annex F.10.1.4 at infinities
    inf = math.inf
    assert bin_op("atan2", [1.0, -1.0, 1.0, inf, inf, -inf], [inf, inf, -inf, 1.0, inf, -inf], "f64", oracle).tolist() == \
        [0.0, -0.0, math.pi, math.pi / 2, math.pi / 4, -3 * math.pi / 4]


def test_pow_against_true_powers_and_annex_f(oracle):
    rng = np.random.default_rng(3)
    a, b = rng.uniform(0.1, 10, 64), rng.uniform(-5, 5, 64)
    got = bin_op("pow", a, b, "f64", oracle)
    want = np.array([float(mp.power(mp.mpf(float(x)), mp.mpf(float(y)))) for x, y in zip(a, b)])
    assert (np.abs(got - want) <= 4 * np.spacing(np.abs(want))).all()
    assert bin_op("pow", [-2.0, -2.0, -8.0], [3.0, 2.0, -1.0], "f64", oracle).tolist() == [-8.0, 4.0, -0.125]
    # integer operands: exact integer power, wrapped to the type (binary_backend.ex:736; shared.ex:190-194)
    i = Nx.pow(from_numpy(np.array([3, -3, 2, 7], dtype=np.int32), "s32", oracle), from_numpy(np.array([5, 3, 31, 20], dtype=np.int32), "s32", oracle))
    assert raw(i).tolist() == [243, -27, -2 ** 31, ((7 ** 20 + 2 ** 31) % 2 ** 32) - 2 ** 31]


def test_divide_and_remainder_on_finite_operands(oracle):
    rng = np.random.default_rng(4)
    a, b = rng.uniform(-100, 100, 64), rng.uniform(0.5, 7, 64) * rng.choice([-1, 1], 64)
    assert np.array_equal(bin_op("divide", a, b, "f64", oracle), a / b)  # IEEE division is correctly rounded: one answer
    r = bin_op("remainder", a, b, "f64", oracle)
    # fmod: exact, the sign of the dividend, |r| < |b|, and a - r is a multiple of b
    assert np.array_equal(r, np.fmod(a, b)) and (np.abs(r) < np.abs(b)).all() and (np.sign(r) * np.sign(a) >= 0).all()
    q = (a - r) / b
    assert np.abs(q - np.round(q)).max() < 1e-9
    # integers: rem/2 keeps the dividend's sign; quotient truncates
    ia, ib = np.array([7, -7, 7, -7], dtype=np.int32), np.array([2, 2, -2, -2], dtype=np.int32)
    assert raw(Nx.remainder(from_numpy(ia, "s32", oracle), from_numpy(ib, "s32", oracle))).tolist() == [1, -1, 1, -1]
    assert raw(Nx.quotient(from_numpy(ia, "s32", oracle), from_numpy(ib, "s32", oracle))).tolist() == [3, -3, -3, 3]
