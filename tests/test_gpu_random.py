"""`Nx.Random` on the device: the reference's known answers through the C ABI, and the device
against the oracle on shapes past the doctests.  Bits, integers and uniform floats are integer
and exactly-rounded float work: bit-exact.  Normal samples pass through log and sqrt in f64, where
the device's math library and the host's may differ in the last place: compared within 4 ulp of
the output type there (the known answers are still met bit for bit)."""
import numpy as np
import pytest

from nx_amd import nx as Nx
from nx_amd import random as Random
from random_support import CASES, check_random_case
from support import assert_all_close, assert_bits_equal, from_numpy, seed_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", CASES, ids=[c["name"] for c in CASES])
def test_device_matches_reference_random_known_answer(case, hip):
    check_random_case(case, hip)


def keys(seed, hip, oracle):
    return Random.key(seed, backend=hip), Random.key(seed, backend=oracle)


@pytest.mark.parametrize("shape", [(), (1,), (7,), (8,), (3, 5), (1001,), (64, 129), (2, 3, 4, 5)])
@pytest.mark.parametrize("bit_width", [8, 16, 32, 64])
def test_random_bits(shape, bit_width, hip, oracle):
    hk, ok = keys(seed_of(shape, bit_width), hip, oracle)
    got = Random.random_bits(hk, shape=shape, bit_width=bit_width)
    assert type(got.data) is hip
    assert_bits_equal(got, Random.random_bits(ok, shape=shape, bit_width=bit_width), f"random_bits {shape} {bit_width}")


@pytest.mark.parametrize("parts", [1, 2, 3, 16, 1000])
def test_split_and_fold_in(parts, hip, oracle):
    hk, ok = keys(parts * 7919, hip, oracle)
    assert_bits_equal(Random.split(hk, parts=parts), Random.split(ok, parts=parts), f"split {parts}")
    data = np.arange(parts * 3, dtype=np.int64).reshape(parts, 3) * 2654435761
    assert_bits_equal(Random.fold_in(hk, Nx.tensor(data, backend=hip)), Random.fold_in(ok, Nx.tensor(data, backend=oracle)),
                      f"fold_in {parts}")


@pytest.mark.parametrize("ty", ["u8", "s8", "u16", "s16", "u32", "s32", "u64", "s64"])
@pytest.mark.parametrize("lo,hi", [(0, 10), (-100, 100), (3, 4), (0, 127)])
def test_randint(ty, lo, hi, hip, oracle):
    if ty.startswith("u") and lo < 0:
        lo, hi = 0, hi - lo
    if hi > 127 and ty.endswith("8") and ty[0] == "s":
        hi = 127
    hk, ok = keys(seed_of(ty, lo, hi), hip, oracle)
    got, hk2 = Random.randint(hk, lo, hi, shape=(37, 11), type=ty)
    want, ok2 = Random.randint(ok, lo, hi, shape=(37, 11), type=ty)
    assert_bits_equal(got, want, f"randint {ty} [{lo}, {hi})")
    assert_bits_equal(hk2, ok2, "randint new key")
    vals = hip.to_numpy(got)
    assert vals.min() >= lo and vals.max() < hi


@pytest.mark.parametrize("ty", ["bf16", "f16", "f32", "f64"])
@pytest.mark.parametrize("lo,hi", [(0.0, 1.0), (-3.5, 12.25), (10, 15)])
def test_uniform(ty, lo, hi, hip, oracle):
    hk, ok = keys(seed_of(ty, lo, hi), hip, oracle)
    got, _ = Random.uniform(hk, lo, hi, shape=(1000, 7), type=ty)
    want, _ = Random.uniform(ok, lo, hi, shape=(1000, 7), type=ty)
    assert_bits_equal(got, want, f"uniform {ty} [{lo}, {hi})")


@pytest.mark.parametrize("ty,ulp", [("bf16", 2.0 ** -8), ("f16", 2.0 ** -11), ("f32", 2.0 ** -24), ("f64", 2.0 ** -53)])
def test_normal(ty, ulp, hip, oracle):
    hk, ok = keys(1337, hip, oracle)
    got, _ = Random.normal(hk, 10, 5, shape=(1000,), type=ty)
    want, _ = Random.normal(ok, 10, 5, shape=(1000,), type=ty)
    assert_all_close(got, want, 4 * ulp, 4 * ulp, f"normal {ty}")
    literal, _ = Random.normal(hk, shape=(512,), type=ty)
    assert_all_close(literal, Random.normal(ok, shape=(512,), type=ty)[0], 4 * ulp, 4 * ulp, f"normal literal {ty}")


def test_moments_of_a_large_sample_stay_on_the_device(hip):
    # nx/test/nx/random_test.exs:259-297: mean and variance of 10000 draws within 10 %
    key = Random.key(1234, backend=hip)
    u = Random.uniform_split(key, 10, 15, shape=(10000,))
    assert type(u.data) is hip
    vals = hip.to_numpy(u).astype(np.float64)
    assert abs(vals.mean() - 12.5) < 0.125 and abs(vals.var() - 25 / 12) < 0.21
    r = hip.to_numpy(Random.randint_split(key, 10, 95, shape=(10000,))).astype(np.float64)
    assert abs(r.mean() - 52.5) < 5.25 and abs(r.var() - 84 * 86 / 12) < 60.2
    n = hip.to_numpy(Random.normal_split(key, 10, 5, shape=(10000,))).astype(np.float64)
    assert abs(n.mean() - 10) < 1 and abs(n.std() - 5) < 0.5


@pytest.mark.parametrize("shape", [(), (1,), (2,), (7,), (8,), (3, 5), (1001,), (64, 129), (1 << 20,), ((1 << 20) + 1,)])
def test_fused_threefry_matches_the_composition(shape, hip):
    key = Random.key(seed_of(shape), backend=hip)
    fused = Random.threefry2x32(key, shape)
    previous = Random.compose_only(True)
    try:
        composed = Random.threefry2x32(key, shape)
    finally:
        Random.compose_only(previous)
    assert_bits_equal(fused, composed, f"threefry2x32 {shape}")


def test_known_answers_hold_through_the_composition_too(hip):
    previous = Random.compose_only(True)
    try:
        for case in CASES:
            check_random_case(case, hip)
    finally:
        Random.compose_only(previous)


# a lane has two vectors of eight words: one, less and more than a lane's, halves off the vector grid, several trips of the grid
@pytest.mark.parametrize("shape", [(1,), (2,), (7,), (15,), (16,), (17,), (33, 31), (4096,), (100003,), (1 << 24,)])
def test_words_made_inside_a_compiled_group(shape, hip):
    """A traced sample makes its words where it uses them and derives its key there: two launches, the bits of the separate calls."""
    from nx_amd import defn
    key = Random.key(20 + len(shape) + shape[0], backend=hip)
    other = from_numpy(np.linspace(-1, 1, int(np.prod(shape)), dtype=np.float32).reshape(shape), "f32", hip)
    functions = {"normal": lambda k, o: Random.normal(k, shape=shape), "uniform": lambda k, o: Random.uniform(k, -2.0, 3.0, shape=shape),
                 "noisy": lambda k, o: Nx.add(o, Nx.multiply(0.25, Random.normal_split(k, shape=shape))),
                 "bits": lambda k, o: Nx.bitwise_xor(Nx.right_shift(Random.random_bits(k, shape=shape), 3), 12345),
                 "third of five": lambda k, o: Random.uniform_split(Random._at(Random.split(k, 5), 2), shape=shape)}
    for name, fun in functions.items():
        planned = defn.compile(fun, key, other, fuse="compiled")
        group = next(r.data.args[0] for r in planned.roots if r.data.op == "fused")
        assert group.words is not None or shape == (1,), name
        calls = []
        original = hip.threefry2x32.__func__
        hip.threefry2x32 = classmethod(lambda cls, *a: (calls.append(1), original(cls, *a))[1])
        try:
            got = planned._evaluate([key, other])
        finally:
            hip.threefry2x32 = classmethod(original)
        assert not calls or shape == (1,), name
        for g, w in zip(got, defn.compile(fun, key, other)._walk([key, other])):
            assert_bits_equal(g, w, f"{name} {shape}")


# The sample and the key for the next one, in one launch where the split's other part is what is asked for
@pytest.mark.parametrize("count", [2, 7, 8, 513, 70001])
@pytest.mark.parametrize("order", ["sample first", "key first", "both keys", "three parts"])
def test_a_sample_and_the_next_key_of_one_split(count, order, hip):
    from nx_amd import defn
    from nx_amd import random as Random

    def program(key):
        keys = Random.split(key, 3 if order == "three parts" else 2)
        sample, after = Random.normal_split(Nx.squeeze(Nx.slice(keys, [1, 0], [1, 2]), axes=[0]), shape=(count,)), Nx.squeeze(Nx.slice(keys, [0, 0], [1, 2]), axes=[0])
        if order == "key first":
            return after, sample
        return (sample, after, Nx.squeeze(Nx.slice(keys, [1, 0], [1, 2]), axes=[0])) if order == "both keys" else (sample, after)
    key = Random.key(2024 + count, backend=hip)
    planned = defn.compile(program, key, fuse="compiled")
    group = next(r.data.args[0] for r in planned.roots if r.data.op == "fused")
    assert group.words is not None and group.beside is not None
    want = [Nx.to_binary(t) for t in program(key)]
    beside, keys = [], []
    fused, random_key = hip.fused_elementwise.__func__, hip.random_key.__func__
    hip.fused_elementwise = classmethod(lambda cls, *a, **k: (beside.append(k.get("beside") is not None), fused(cls, *a, **k))[1])
    hip.random_key = classmethod(lambda cls, *a: (keys.append(a[3]), random_key(cls, *a))[1])
    try:
        assert [Nx.to_binary(t) for t in planned._walk([key])] == want
    finally:
        hip.fused_elementwise, hip.random_key = classmethod(fused), classmethod(random_key)
    # a key that is there before the sample is not made again; one that is the sample's own is never beside it
    assert beside == [order != "key first"] and keys == {"key first": [0], "both keys": [1]}.get(order, [])
    for _ in range(5):  # (evaluated, recorded, issued from the recording)
        assert [Nx.to_binary(t) for t in planned(key)] == want
