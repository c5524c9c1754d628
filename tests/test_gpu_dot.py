"""Device Nx.dot against the CPU oracle.

Bar: integer results bit-exact (s8 x s8 -> s32 / s8 on MFMA, everything else on the plain
kernel); float results within the K-scaled bound
    |d| <= 2K * 2^-24 * sum_k |a_k b_k|  +  1 ulp(out type) * |ref|
(the device accumulates in f32 on MFMA, the reference sequentially in f64), and for f64 operands
within 1e-13 relative to sum|a_k b_k|."""
import numpy as np
import pytest

from nx_amd import nx as Nx
from nx_amd import types as T
from support import assert_bits_equal, from_numpy, seed_of, values
from test_gpu_elementwise import both, rand_raw

pytestmark = pytest.mark.gpu

ULP = {("bf", 16): 2.0 ** -7, ("f", 16): 2.0 ** -10, ("f", 32): 2.0 ** -23, ("f", 64): 2.0 ** -52}


def check_float_dot(got, want, a64, b64, eq, K, what):
    """a64/b64: decoded operands; eq: einsum spec producing the output from |a|, |b|."""
    assert got.type == want.type and got.shape == want.shape, what
    mag = np.einsum(eq, np.abs(a64), np.abs(b64)).reshape(got.shape)
    ref = values(want)
    acc = 2.0 ** -24 if got.type != ("f", 64) and True else 2.0 ** -50
    bound = 2 * max(K, 1) * acc * mag + ULP[got.type] * np.abs(ref) + 1e-30
    err = np.abs(values(got) - ref)
    assert (err <= bound).all(), f"{what}: max err/bound {np.max(err / bound):.3f}"


MNK = [(128, 128, 64), (256, 256, 256), (130, 70, 136), (1, 1, 8), (17, 300, 1000), (512, 64, 2048), (64, 11008 // 8, 4096),
       (33, 33, 40), (200, 129, 8), (5, 7, 3), (64, 64, 7)]


@pytest.mark.parametrize("M,N,K", MNK)
@pytest.mark.parametrize("ty", ["bf16", "f16", "f32", "f64"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_float_matmul_layouts(M, N, K, ty, layout, hip, oracle):
    if ty == "f64" and M * N * K > 5_000_000:
        pytest.skip("plain-kernel path: covered at smaller sizes")
    rng = np.random.default_rng(seed_of(M, N, K, ty))
    a_shape = (M, K) if layout[0] == "n" else (K, M)
    b_shape = (K, N) if layout[1] == "n" else (N, K)
    a, b = rand_raw(rng, ty, a_shape, lo=-1, hi=1), rand_raw(rng, ty, b_shape, lo=-1, hi=1)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    got, want = Nx.dot(ha, c1, hb, c2), Nx.dot(oa, c1, ob, c2)
    eq = ("mk" if layout[0] == "n" else "km") + "," + ("kn" if layout[1] == "n" else "nk") + "->mn"
    check_float_dot(got, want, values(oa), values(ob), eq, K, f"dot {ty} {layout} {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(64, 344, 4096), (128, 128, 128), (7, 9, 16), (130, 70, 1024), (64, 64, 48), (3, 5, 7)])
@pytest.mark.parametrize("out_type", ["s32", "s8", "s64"])
def test_int8_dot_is_bit_exact(M, N, K, out_type, hip, oracle):
    rng = np.random.default_rng(seed_of(M, N, K))
    x = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
    w = rng.integers(-127, 128, size=(N, K)).astype(np.int8)
    hx, ox = both(x, "s8", hip, oracle)
    hw, ow = both(w, "s8", hip, oracle)
    ot = None if out_type == "s8" else out_type  # s8 is what the public API infers (wraps)
    assert_bits_equal(Nx.dot(hx, [1], hw, [1], out_type=ot), Nx.dot(ox, [1], ow, [1], out_type=ot), f"s8 dot -> {out_type}")
    # exact closed form as an independent check of both
    exact = x.astype(np.int64) @ w.astype(np.int64).T
    got = hip.to_numpy(Nx.dot(hx, [1], hw, [1], out_type="s32"))
    assert np.array_equal(got, exact.astype(np.int32))


@pytest.mark.parametrize("lt,rt", [("s32", "s32"), ("u8", "u8"), ("s16", "s64"), ("u32", "s8"), ("s64", "s64"), ("u8", "s8")])
def test_integer_dot_is_bit_exact(lt, rt, hip, oracle):
    rng = np.random.default_rng(seed_of(lt, rt))
    a, b = rand_raw(rng, lt, (19, 45)), rand_raw(rng, rt, (45, 23))
    ha, oa = both(a, lt, hip, oracle)
    hb, ob = both(b, rt, hip, oracle)
    assert_bits_equal(Nx.dot(ha, hb), Nx.dot(oa, ob), f"dot {lt} {rt}")


@pytest.mark.parametrize("lt,rt", [("f32", "bf16"), ("s8", "f32"), ("f16", "f32"), ("f64", "f32")])
def test_mixed_type_dot(lt, rt, hip, oracle):
    rng = np.random.default_rng(seed_of(lt, rt))
    a, b = rand_raw(rng, lt, (40, 64), lo=-1, hi=1), rand_raw(rng, rt, (64, 24), lo=-1, hi=1)
    ha, oa = both(a, lt, hip, oracle)
    hb, ob = both(b, rt, hip, oracle)
    check_float_dot(Nx.dot(ha, hb), Nx.dot(oa, ob), values(oa), values(ob), "mk,kn->mn", 64, f"dot {lt} {rt}")


BATCHED = [((32, 64, 64), [2], [0], (32, 48, 64), [2], [0], "bmk,bnk->bmn"),
           ((4, 16, 40), [1], [0], (4, 16, 24), [1], [0], "bkm,bkn->bmn"),
           ((3, 5, 32, 8), [3], [0, 1], (3, 5, 8, 16), [2], [0, 1], "abmk,abkn->abmn"),
           ((2, 8, 16, 4), [1, 3], [0], (2, 4, 8, 6), [2, 1], [0], "bkml,blkn->bmn"),
           ((6, 10), [0, 1], [], (10, 6), [1, 0], [], "ab,ba->"),
           ((4, 6, 5), [1], [], (3, 6, 2), [1], [], "amb,cmd->abcd"),
           ((8, 3), [], [], (2, 5), [], [], "ab,cd->abcd")]


@pytest.mark.parametrize("case", BATCHED, ids=[c[-1] for c in BATCHED])
@pytest.mark.parametrize("ty", ["bf16", "f32", "s32", "s8"])
def test_general_contraction_and_batch_axes(case, ty, hip, oracle):
    ls, c1, b1, rs, c2, b2, eq = case
    rng = np.random.default_rng(seed_of(eq, ty))
    a, b = rand_raw(rng, ty, ls, lo=-1, hi=1), rand_raw(rng, ty, rs, lo=-1, hi=1)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    got, want = Nx.dot(ha, c1, b1, hb, c2, b2), Nx.dot(oa, c1, b1, ob, c2, b2)
    if T.is_integer(T.normalize(ty)):
        assert_bits_equal(got, want, f"dot {eq} {ty}")
    else:
        K = int(np.prod([ls[x] for x in c1])) if c1 else 1
        check_float_dot(got, want, values(oa), values(ob), eq, K, f"dot {eq} {ty}")


def test_dot_matches_closed_form_on_small_integers_in_bf16(hip):
    """Small-integer operands make every partial sum exact in f32: the MFMA result must equal the
    integer matrix product exactly, whatever the accumulation order."""
    rng = np.random.default_rng(2)
    a = rng.integers(-4, 5, size=(256, 512))
    b = rng.integers(-4, 5, size=(512, 384))
    bits = lambda m: (m.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    ha, hb = from_numpy(bits(a), "bf16", hip), from_numpy(bits(b), "bf16", hip)
    got = values(Nx.dot(Nx.as_type(ha, "f32"), Nx.as_type(hb, "f32")))
    assert np.array_equal(got, (a @ b).astype(np.float64))
    got_bf = values(Nx.dot(ha, hb, out_type="f32"))
    assert np.array_equal(got_bf, (a @ b).astype(np.float64))


@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (64, 48, 128), (130, 72, 256), (512, 528, 384), (16, 4096, 128)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_int8_dot_every_operand_layout_is_bit_exact(M, N, K, layout, hip, oracle):
    """K-outer s8 operands are transposed inside the MFMA kernel (or by a pass when the row count
    is ragged): all four layouts must give the exact integer product."""
    rng = np.random.default_rng(seed_of(M, N, K, layout))
    a = rng.integers(-128, 128, size=(M, K) if layout[0] == "n" else (K, M)).astype(np.int8)
    b = rng.integers(-128, 128, size=(K, N) if layout[1] == "n" else (N, K)).astype(np.int8)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    got = hip.to_numpy(Nx.dot(from_numpy(a, "s8", hip), c1, from_numpy(b, "s8", hip), c2, out_type="s32"))
    am = a if layout[0] == "n" else a.T
    bm = b if layout[1] == "n" else b.T
    exact = (am.astype(np.float64) @ bm.astype(np.float64)).astype(np.int64)  # exact: |sum| < 2^53
    assert np.array_equal(got, exact.astype(np.int32))
    want = Nx.dot(from_numpy(a, "s8", oracle), c1, from_numpy(b, "s8", oracle), c2, out_type="s32")
    assert np.array_equal(got, np.frombuffer(Nx.to_binary(want), dtype=np.int32).reshape(M, N))


@pytest.mark.parametrize("ty,M,N,K", [("f32", 128, 128, 64), ("f32", 100, 36, 96), ("f32", 102, 38, 96), ("bf16", 136, 72, 128),
                                      ("f16", 264, 200, 192), ("bf16", 132, 76, 64), ("f32", 300, 260, 2048)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_float_dot_pipelined_kernel_layouts(ty, M, N, K, layout, hip, oracle):
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout))
    a = rand_raw(rng, ty, (M, K) if layout[0] == "n" else (K, M), lo=-1, hi=1)
    b = rand_raw(rng, ty, (K, N) if layout[1] == "n" else (N, K), lo=-1, hi=1)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    eq = ("mk" if layout[0] == "n" else "km") + "," + ("kn" if layout[1] == "n" else "nk") + "->mn"
    check_float_dot(Nx.dot(ha, c1, hb, c2), Nx.dot(oa, c1, ob, c2), values(oa), values(ob), eq, K, f"{ty} {layout} {M}x{N}x{K}")


# Few rows against a long K-inner matrix (M <= 64, K a multiple of 4096 bytes, N >= 256) take
# the weight-streaming kernel: ragged row counts, a column count that is not a multiple of the
# 64 columns of a work-group, every MFMA element type, and a batch.
@pytest.mark.parametrize("M", [1, 16, 33, 64])
@pytest.mark.parametrize("ty,N,K", [("s8", 300, 4096), ("s8", 1000, 8192), ("bf16", 264, 2048), ("f16", 257, 4096),
                                    ("f32", 320, 1024), ("bf16", 1024, 4096)])
def test_few_rows_against_long_matrix(M, ty, N, K, hip, oracle):
    rng = np.random.default_rng(seed_of(M, ty, N, K))
    if ty == "s8":
        x = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        w = rng.integers(-127, 128, size=(N, K)).astype(np.int8)
        hx, ox = both(x, ty, hip, oracle)
        hw, ow = both(w, ty, hip, oracle)
        got, want = Nx.dot(hx, [1], hw, [1], out_type="s32"), Nx.dot(ox, [1], ow, [1], out_type="s32")
        assert_bits_equal(got, want, f"few rows s8 {M}x{N}x{K}")
    else:
        x, w = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (N, K), lo=-1, hi=1)
        hx, ox = both(x, ty, hip, oracle)
        hw, ow = both(w, ty, hip, oracle)
        got, want = Nx.dot(hx, [1], hw, [1]), Nx.dot(ox, [1], ow, [1])
        check_float_dot(got, want, values(ox), values(ow), "mk,nk->mn", K, f"few rows {ty} {M}x{N}x{K}")


@pytest.mark.parametrize("M", [1, 24, 64])
@pytest.mark.parametrize("ty,N,K", [("bf16", 264, 2048), ("f16", 1024, 1056), ("s8", 400, 4096), ("bf16", 120, 640), ("bf16", 328, 192),
                                    ("s8", 12304, 1152), ("s8", 1040, 1024), ("s8", 48, 2048)])
def test_few_rows_against_weights_stored_k_outer(M, ty, N, K, hip, oracle):
    """x . W with W stored [K, N], the plain Nx.dot(x, w): a few rows of a 2-byte type take the 128-row kernels
    (which read a K-outer operand by transposing loads, K split over work-groups when long), int8 the 64-row tiles
    with 64 or -- for many columns -- 128 columns of the weights, read by the byte-transposing loads; a contraction
    length that is an odd number of slabs takes one slab per phase."""
    rng = np.random.default_rng(seed_of(M, ty, N, K, "k-outer weights"))
    if ty == "s8":
        x = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        w = rng.integers(-127, 128, size=(K, N)).astype(np.int8)
        hx, ox = both(x, ty, hip, oracle)
        hw, ow = both(w, ty, hip, oracle)
        assert_bits_equal(Nx.dot(hx, hw, out_type="s32"), Nx.dot(ox, ow, out_type="s32"), f"few rows s8 {M}x{N}x{K} NN")
    else:
        x, w = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
        hx, ox = both(x, ty, hip, oracle)
        hw, ow = both(w, ty, hip, oracle)
        check_float_dot(Nx.dot(hx, hw), Nx.dot(ox, ow), values(ox), values(ow), "mk,kn->mn", K, f"few rows {ty} {M}x{N}x{K} NN")


@pytest.mark.parametrize("ty,M,N,K", [("bf16", 64, 1024, 1152), ("s8", 33, 520, 1152), ("f16", 7, 300, 4224), ("s8", 64, 11008, 4096)])
def test_few_rows_one_and_two_slabs_per_phase(ty, M, N, K, hip, oracle):
    """K-inner operands on 64 x 64 tiles of the two-group kernel: K of an odd number of slabs walks one slab per
    phase through eight stages, an even number two per phase through four."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, "rows phases"))
    if ty == "s8":
        x = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        w = rng.integers(-127, 128, size=(N, K)).astype(np.int8)
        got = hip.to_numpy(Nx.dot(from_numpy(x, ty, hip), [1], from_numpy(w, ty, hip), [1], out_type="s32"))
        assert np.array_equal(got, x.astype(np.int32) @ w.astype(np.int32).T)
    else:
        x, w = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (N, K), lo=-1, hi=1)
        hx, ox = both(x, ty, hip, oracle)
        hw, ow = both(w, ty, hip, oracle)
        check_float_dot(Nx.dot(hx, [1], hw, [1]), Nx.dot(ox, [1], ow, [1]), values(ox), values(ow), "mk,nk->mn", K, f"few rows {ty} {M}x{N}x{K}")


def test_few_rows_against_long_matrix_batched(hip, oracle):
    rng = np.random.default_rng(7)
    x = rng.integers(-127, 128, size=(3, 20, 4096)).astype(np.int8)
    w = rng.integers(-127, 128, size=(3, 272, 4096)).astype(np.int8)
    hx, ox = both(x, "s8", hip, oracle)
    hw, ow = both(w, "s8", hip, oracle)
    got = Nx.dot(hx, [2], [0], hw, [2], [0], out_type="s32")
    want = Nx.dot(ox, [2], [0], ow, [2], [0], out_type="s32")
    assert_bits_equal(got, want, "few rows s8 batched")


# Shapes large enough for the 256 x 256 tile (at least 192 of them), ragged at both edges, in every
# operand layout: covers the transposing-read staging of K-outer bf16 and s8 operands on both
# sides.  The oracle runs on a sample of output rows.
@pytest.mark.parametrize("ty", ["bf16", "s8"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_large_ragged_dot_on_the_big_tile(ty, layout, hip, oracle):
    M, N, K = 2064, 6160, 256
    rng = np.random.default_rng(seed_of(ty, layout, "big tile"))
    if ty == "s8":
        a = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        b = rng.integers(-127, 128, size=(K, N)).astype(np.int8)
    else:
        a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    kw = {"out_type": "s32"} if ty == "s8" else {}
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2, **kw)
    assert got.shape == (M, N)
    rows = np.unique(np.concatenate([[0, 255, 256, M - 1], rng.integers(0, M, size=24)]))
    oa, ob = from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle)
    want = Nx.dot(oa, ob, **kw)
    got_rows = from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), "s32" if ty == "s8" else ty, oracle)
    if ty == "s8":
        assert_bits_equal(got_rows, want, f"big tile s8 {layout}")
    else:
        check_float_dot(got_rows, want, values(oa), values(ob), "mk,kn->mn", K, f"big tile {ty} {layout}")


@pytest.mark.parametrize("ty", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(1024, 6144, 256), (1000, 6200, 384), (2048, 3080, 128)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_half_width_tiles_of_the_two_group_kernel(ty, M, N, K, layout, hip, oracle):
    """Problems whose grid of 256 x 256 tiles would leave CUs idle take 256 x 128 tiles (wave tiles 64 x 64 or
    128 x 32): whole and ragged grids, all four operand layouts."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "w128"))
    a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2)
    assert got.shape == (M, N)
    rows = np.unique(np.concatenate([[0, 127, 128, 255, 256, M - 1], rng.integers(0, M, size=18)]))
    oa, ob = from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle)
    want = Nx.dot(oa, ob)
    got_rows = from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), ty, oracle)
    check_float_dot(got_rows, want, values(oa), values(ob), "mk,kn->mn", K, f"256x128 tiles {ty} {layout}")


@pytest.mark.parametrize("ty,M,N,K", [("bf16", 333, 777, 555), ("f16", 256, 512, 1000), ("f32", 300, 260, 250), ("s8", 384, 320, 1001),
                                      ("bf16", 2, 4100, 2050)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_contraction_lengths_off_the_slab_grid_are_padded(ty, M, N, K, layout, hip, oracle):
    """A K that is not a whole number of 128-byte slabs: the partial slab is walked in place with zeros behind its end
    (K-inner rows that are not whole 16-byte pieces are first copied to rows that are), and products of two zeros add
    nothing: int8 stays exact and floats stay within the bound."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "pad"))
    if ty == "s8":
        a = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        b = rng.integers(-127, 128, size=(K, N)).astype(np.int8)
    else:
        a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    kw = {"out_type": "s32"} if ty == "s8" else {}
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2, **kw)
    assert got.shape == (M, N)
    rows = np.unique(np.concatenate([[0, M - 1], rng.integers(0, M, size=10)]))
    oa, ob = from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle)
    want = Nx.dot(oa, ob, **kw)
    got_rows = from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), "s32" if ty == "s8" else ty, oracle)
    if ty == "s8":
        assert_bits_equal(got_rows, want, f"padded K s8 {layout}")
    else:
        check_float_dot(got_rows, want, values(oa), values(ob), "mk,kn->mn", K, f"padded K {ty} {layout}")


# The partial slab of K in every kernel that walks slabs: one piece or one k of it, all but one, nothing but a partial
# slab, an odd number of slabs, K split over work-groups so that the last range is shorter and holds it.
@pytest.mark.parametrize("ty,M,N,K", [("bf16", 2064, 6160, 72), ("f16", 1000, 6200, 1), ("bf16", 2048, 3080, 191), ("bf16", 520, 392, 1032),
                                      ("f16", 40, 1024, 1160), ("bf16", 24, 2048, 648), ("bf16", 128, 1024, 4104), ("bf16", 96, 392, 63),
                                      ("f32", 300, 264, 36), ("f32", 1024, 512, 785), ("f32", 512, 10, 4092), ("f32", 40, 384, 1001),
                                      ("s8", 2064, 6160, 144), ("s8", 64, 12304, 1168), ("s8", 48, 272, 1297), ("s8", 130, 528, 4112), ("s8", 256, 256, 5)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_partial_slabs_of_k(ty, M, N, K, layout, hip):
    """Integer-valued operands: every partial sum is a whole number below 2^24 (4 * 4 * 5000), so each order of
    additions gives the exact product in f32 and s32 alike."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "partial slab"))
    a, b = rng.integers(-4, 5, size=(M, K)), rng.integers(-4, 5, size=(K, N))
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    held = {"s8": lambda x: x.astype(np.int8), "f32": lambda x: x.astype(np.float32), "f16": lambda x: x.astype(np.float16),
            "bf16": lambda x: (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)}[ty]
    out = "s32" if ty == "s8" else "f32"
    got = Nx.dot(from_numpy(held(la), ty, hip), [1 if layout[0] == "n" else 0], from_numpy(held(lb), ty, hip),
                 [0 if layout[1] == "n" else 1], out_type=out)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.int32 if ty == "s8" else np.float32)
    assert np.array_equal(hip.to_numpy(got), want)


HELD = {"s8": lambda x: x.astype(np.int8), "f32": lambda x: x.astype(np.float32), "f16": lambda x: x.astype(np.float16),
        "f64": lambda x: x.astype(np.float64), "bf16": lambda x: (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)}


# every copy with a batch: K-inner rows padded, K-outer ones re-laid and padded, one operand copied and the other not, none copied
@pytest.mark.parametrize("ty,batch,M,N,K", [("bf16", 5, 203, 197, 333), ("bf16", 3, 264, 197, 333), ("f16", 3, 264, 520, 72), ("f32", 4, 160, 131, 250),
                                            ("s8", 3, 256, 272, 301), ("s8", 2, 130, 528, 1297)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_batched_contractions_with_a_partial_slab(ty, batch, M, N, K, layout, hip):
    """Integer-valued operands: every partial sum is a whole number below 2^24, so the product is exact in any order."""
    rng = np.random.default_rng(seed_of(ty, batch, M, N, K, layout, "batched partial slab"))
    a, b = rng.integers(-4, 5, size=(batch, M, K)), rng.integers(-4, 5, size=(batch, K, N))
    la = a if layout[0] == "n" else np.ascontiguousarray(a.transpose(0, 2, 1))
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.transpose(0, 2, 1))
    got = Nx.dot(from_numpy(HELD[ty](la), ty, hip), [2 if layout[0] == "n" else 1], [0], from_numpy(HELD[ty](lb), ty, hip),
                 [1 if layout[1] == "n" else 2], [0], out_type="s32" if ty == "s8" else "f32")
    assert np.array_equal(hip.to_numpy(got).astype(np.float64), a.astype(np.float64) @ b.astype(np.float64))


@pytest.mark.parametrize("ty,M,N,K", [("bf16", 264, 520, 72), ("f16", 520, 392, 1032), ("bf16", 24, 2048, 648), ("bf16", 203, 264, 333),
                                      ("f32", 132, 64, 36), ("f32", 300, 264, 250)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_what_lies_behind_the_end_of_k_is_not_read(ty, M, N, K, layout, hip):
    """NaN in the next row, the next column, the next batch item and behind the operands: it stays out of the results of
    the others, which are exact (integer-valued operands)."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "behind the end"))
    a, b = rng.integers(-4, 5, size=(3, M, K)).astype(np.float64), rng.integers(-4, 5, size=(3, K, N)).astype(np.float64)
    a[1], b[2] = np.nan, np.nan
    a[0, 1::2], b[0, :, 2::3] = np.nan, np.inf
    la = a if layout[0] == "n" else np.ascontiguousarray(a.transpose(0, 2, 1))
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.transpose(0, 2, 1))

    def followed_by_nan(x):
        held = HELD[ty](x)
        nan = HELD[ty](np.full(256, np.nan))
        owner = from_numpy(np.concatenate([held.ravel(), nan]), ty, hip)
        pointer = Nx.Pointer(kind="local", address=Nx.to_pointer(owner).address, data_size=held.size * held.itemsize)
        return Nx.from_pointer(hip, pointer, ty, held.shape, keep=owner)
    got = hip.to_numpy(Nx.dot(followed_by_nan(la), [2 if layout[0] == "n" else 1], [0], followed_by_nan(lb), [1 if layout[1] == "n" else 2], [0],
                              out_type="f32")).astype(np.float64)
    want = a[0, ::2] @ np.nan_to_num(b[0], posinf=0.0)
    finite = np.arange(N) % 3 != 2
    assert np.array_equal(got[0, ::2][:, finite], want[:, finite])
    assert np.isnan(got[0, 1::2]).all() and not np.isfinite(got[0, ::2][:, ~finite]).any() and np.isnan(got[1:]).all()


# Rows and k-rows one element longer or shorter than whole 16-byte pieces, in every kernel: the smallest operands the matrix
# kernels take, few rows, 32- to 256-row tiles, K split, whole slabs of K under a k-row that is not whole pieces.
@pytest.mark.parametrize("ty,M,N,K", [("s8", 17, 17, 17), ("s8", 33, 31, 15), ("s8", 7, 1057, 296), ("s8", 43, 379, 2049), ("s8", 65, 4097, 1024),
                                      ("s8", 271, 130, 129), ("s8", 1025, 2063, 640), ("bf16", 9, 20, 64), ("bf16", 1, 1031, 2047), ("bf16", 31, 1027, 512),
                                      ("f16", 257, 393, 321), ("bf16", 1281, 515, 1093), ("bf16", 2061, 3075, 576), ("f16", 131, 1037, 4097),
                                      ("f32", 21, 13, 32), ("f32", 785, 131, 1025), ("f32", 1021, 10, 1669), ("f32", 66, 515, 992)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_rows_that_are_not_whole_pieces(ty, M, N, K, layout, hip):
    """Integer-valued operands: the product is exact in any order.  What is not a number behind a K-inner operand would show in its
    last row or column if the end of a row were not cut off there; behind a K-outer one it would meet only rows and columns that are not
    stored, whatever is read (that no load leaves either is test_dot_loads.py's)."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "not whole pieces"))
    a, b = rng.integers(-4, 5, size=(M, K)), rng.integers(-4, 5, size=(K, N))
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)

    def followed_by_garbage(x):
        held = HELD[ty](x)
        behind = np.full(256, 77, np.int8) if ty == "s8" else HELD[ty](np.full(256, np.nan))
        owner = from_numpy(np.concatenate([held.ravel(), behind]), ty, hip)
        pointer = Nx.Pointer(kind="local", address=Nx.to_pointer(owner).address, data_size=held.size * held.itemsize)
        return Nx.from_pointer(hip, pointer, ty, held.shape, keep=owner)
    c1, c2 = [1 if layout[0] == "n" else 0], [0 if layout[1] == "n" else 1]
    want = a.astype(np.float64) @ b.astype(np.float64)
    for out in ["s32", "s8"] if ty == "s8" else ["f32", ty]:
        got = Nx.dot(followed_by_garbage(la), c1, followed_by_garbage(lb), c2, out_type=out)
        if out == "s8":
            assert np.array_equal(hip.to_numpy(got), want.astype(np.int64).astype(np.int8))
        elif out == "s32" or ty == "f32":
            assert np.array_equal(hip.to_numpy(got).astype(np.float64), want)
        else:  # rounded once: toward zero in bf16, to nearest in f16
            assert (np.abs(values(got).reshape(M, N) - want) <= ULP[got.type] * np.abs(want)).all()


def at_odd_address(arr, ty, hip, elements):
    """`arr` on the device, `elements` behind the start of an allocation, as a tensor over borrowed memory."""
    flat = np.concatenate([np.zeros(elements, arr.dtype), arr.ravel(), np.zeros(3, arr.dtype)])
    owner = from_numpy(flat, ty, hip)
    size = arr.itemsize
    pointer = Nx.Pointer(kind="local", address=Nx.to_pointer(owner).address + elements * size, data_size=arr.size * size)
    return Nx.from_pointer(hip, pointer, ty, arr.shape, keep=owner)


# every operand form a contraction kernel takes where it lies: whole slabs, a partial slab, rows that are copied anyway, f64
@pytest.mark.parametrize("ty,M,N,K", [("bf16", 264, 520, 128), ("f16", 128, 512, 1032), ("bf16", 24, 2048, 648), ("f32", 132, 64, 36),
                                      ("f32", 300, 264, 250), ("s8", 64, 304, 1168), ("s8", 272, 256, 512), ("f64", 130, 66, 48)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("behind", [(1, 0), (0, 3), (1, 1)])
def test_operands_that_begin_off_a_sixteen_byte_address(ty, M, N, K, layout, behind, hip):
    """Borrowed memory may begin anywhere: the kernels' loads into LDS take their 16 bytes at any address.  Integer-valued
    operands: every partial sum is a whole number below 2^24, so the product is exact in any order."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, behind, "odd address"))
    a, b = rng.integers(-4, 5, size=(M, K)), rng.integers(-4, 5, size=(K, N))
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    left, right = at_odd_address(HELD[ty](la), ty, hip, behind[0]), at_odd_address(HELD[ty](lb), ty, hip, behind[1])
    out = {"s8": "s32", "f64": "f64"}.get(ty, "f32")
    got = Nx.dot(left, [1 if layout[0] == "n" else 0], right, [0 if layout[1] == "n" else 1], out_type=out)
    assert np.array_equal(hip.to_numpy(got).astype(np.float64), a.astype(np.float64) @ b.astype(np.float64))


@pytest.mark.parametrize("ty,M,N,K", [("f32", 64, 48, 33), ("f32", 64, 64, 4095), ("f32", 16, 16, 1001), ("bf16", 128, 96, 1001), ("f16", 64, 64, 4001)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_small_contractions_with_k_off_sixteen_bytes_sum_in_f64_in_every_layout(ty, M, N, K, layout, hip, oracle):
    """A gradient of a layer over a batch of 33 or 4095 rows is dot(x, [0], d, [0]): both operands K-outer.  Below 16 M
    multiply-adds it has the reference's f64 sums, in order of k and rounded once, as the same product stored K-inner has:
    the reference's bits.  (An f32 sum of 33 products of f32 values misses some of 3072 results by a rounding.)"""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "off sixteen bytes"))
    a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1, c2 = [1 if layout[0] == "n" else 0], [0 if layout[1] == "n" else 1]
    ha, oa = both(la, ty, hip, oracle)
    hb, ob = both(lb, ty, hip, oracle)
    assert_bits_equal(Nx.dot(ha, c1, hb, c2, out_type="f32"), Nx.dot(oa, c1, ob, c2, out_type="f32"), f"{ty} {M}x{N}x{K} {layout}")


@pytest.mark.parametrize("ty,M,N,K", [("bf16", 128, 1024, 4096), ("s8", 128, 1024, 4096), ("f16", 200, 520, 2048), ("f32", 132, 384, 2048),
                                      ("bf16", 768, 4096, 4096), ("f16", 1000, 4100, 4096),
                                      ("s8", 384, 512, 8192), ("bf16", 512, 1024, 2048),
                                      # f32 is cut much earlier: 64 ways, two ways with two slabs each, 64 x 32 tiles
                                      ("f32", 256, 264, 4096), ("f32", 128, 128, 128), ("f32", 520, 512, 512), ("f32", 1024, 1024, 1024)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_long_k_on_an_under_filled_grid_is_split(ty, M, N, K, layout, hip, oracle):
    """A few hundred rows against a long K leave most CUs without a 128 x 128 tile; K is then split over
    several work-groups per tile and the partial results are added by a second pass.  int8 must stay exact,
    floats within the bound of an f32 accumulation in any order."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "split"))
    if ty == "s8":
        a = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        b = rng.integers(-127, 128, size=(K, N)).astype(np.int8)
    else:
        a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    kw = {"out_type": "s32"} if ty == "s8" else {}
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2, **kw)
    assert got.shape == (M, N)
    rows = np.unique(np.concatenate([[0, 127, M - 1], rng.integers(0, M, size=13)]))
    oa, ob = from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle)
    want = Nx.dot(oa, ob, **kw)
    got_rows = from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), "s32" if ty == "s8" else ty, oracle)
    if ty == "s8":
        assert_bits_equal(got_rows, want, f"split K s8 {layout}")
    else:
        check_float_dot(got_rows, want, values(oa), values(ob), "mk,kn->mn", K, f"split K {ty} {layout}")


@pytest.mark.parametrize("ty,M,N,K", [("bf16", 512, 520, 256), ("bf16", 300, 528, 128), ("f16", 264, 344, 128), ("bf16", 1024, 6152, 64),
                                      ("bf16", 130, 76, 64), ("f16", 64, 40, 128)])
def test_two_byte_outputs_land_in_their_own_columns(ty, M, N, K, hip):
    """The MFMA kernel writes bf16 / f16 results two column tiles at a time, lanes trading halves
    so that each stores 16 bytes.  A selection matrix (one 1.0 per column) makes every output a
    copy of one input element, so any mix-up of lanes, tiles or columns shows as a wrong value
    -- exact, no tolerance."""
    rng = np.random.default_rng(seed_of(ty, M, N, K))
    a = rand_raw(rng, ty, (M, K), lo=-1, hi=1)
    pick = (7 * np.arange(N) + 3) % K
    b = np.zeros((K, N), dtype=a.dtype)
    b[pick, np.arange(N)] = np.uint16(0x3F80) if ty == "bf16" else np.float16(1.0)
    got = values(Nx.dot(from_numpy(a, ty, hip), from_numpy(b, ty, hip)))
    want = values(from_numpy(np.ascontiguousarray(a[:, pick]), ty, hip))
    assert got.shape == (M, N)
    assert np.array_equal(got, want)  # (-0.0 == 0.0: a lone product plus zeros may lose the sign of a zero)


@pytest.mark.parametrize("ty,M,N,K", [("bf16", 1024, 1024, 1024), ("bf16", 1000, 904, 576), ("f16", 520, 1288, 640), ("bf16", 200, 136, 512),
                                      ("s8", 1024, 1024, 1024), ("s8", 2056, 3080, 1152), ("f16", 2048, 2048, 1088)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_two_groups_sharing_k_on_128_tiles(ty, M, N, K, layout, hip, oracle):
    """Grids of 128 x 128 tiles that fit the CUs once (for int8: any grid, both operands K-inner) are walked by two
    groups of waves that take the even and the odd slabs of K and add their partial sums at the end: even and odd
    numbers of slabs, whole and ragged grids, all four layouts.  int8 exact, floats within the bound."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, layout, "pp128"))
    if ty == "s8":
        a = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        b = rng.integers(-127, 128, size=(K, N)).astype(np.int8)
    else:
        a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    kw = {"out_type": "s32"} if ty == "s8" else {}
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2, **kw)
    assert got.shape == (M, N)
    rows = np.unique(np.concatenate([[0, 31, 32, 63, 64, 127, 128, M - 1], rng.integers(0, M, size=16)]))
    oa, ob = from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle)
    want = Nx.dot(oa, ob, **kw)
    got_rows = from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), "s32" if ty == "s8" else ty, oracle)
    if ty == "s8":
        assert_bits_equal(got_rows, want, f"128 tiles, two groups, s8 {layout}")
    else:
        check_float_dot(got_rows, want, values(oa), values(ob), "mk,kn->mn", K, f"128 tiles, two groups, {ty} {layout}")


@pytest.mark.parametrize("ty,M,N,K,out_type", [("bf16", 1024, 1032, 1024, None), ("f16", 520, 776, 576, None), ("bf16", 768, 512, 640, "f32"),
                                               ("s8", 1024, 520, 1152, "s32"), ("s8", 264, 392, 1024, "s8")])
def test_two_groups_sharing_k_put_every_output_in_its_place(ty, M, N, K, out_type, hip):
    """A selection matrix (a single 1 per column, spread over even and odd slabs) makes every output a copy of one
    input element: a tile half, row or column that ends up with the wrong group shows as a wrong value -- exact."""
    rng = np.random.default_rng(seed_of(ty, M, N, K, "pp128 pick"))
    pick = (37 * np.arange(N) + 11) % K
    if ty == "s8":
        a = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        b = np.zeros((N, K), dtype=np.int8)
        b[np.arange(N), pick] = 1
        got = hip.to_numpy(Nx.dot(from_numpy(a, ty, hip), [1], from_numpy(b, ty, hip), [1], out_type=out_type))
        assert got.shape == (M, N)
        assert np.array_equal(got.astype(np.int64), a[:, pick].astype(np.int64))
        return
    a = rand_raw(rng, ty, (M, K), lo=-1, hi=1)
    b = np.zeros((K, N), dtype=a.dtype)
    b[pick, np.arange(N)] = np.uint16(0x3F80) if ty == "bf16" else np.float16(1.0)
    kw = {"out_type": out_type} if out_type else {}
    got = values(Nx.dot(from_numpy(a, ty, hip), from_numpy(b, ty, hip), **kw))
    want = values(from_numpy(np.ascontiguousarray(a[:, pick]), ty, hip))
    assert got.shape == (M, N)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("M,N,K", [(1, 1, 4096), (1, 1, 70003), (16, 16, 8192), (3, 5, 4100), (32, 1, 5000), (1, 32, 12288), (7, 2, 40000)])
@pytest.mark.parametrize("ty", ["f32", "bf16", "f64", "s8", "s32", "u8"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_few_outputs_over_a_long_contraction(M, N, K, ty, layout, hip, oracle):
    """The dot of two long vectors, a handful of outputs over K >= 4096: a work-group per output and segment of K with
    partial sums in f64 / 64-bit integers and a pass that adds the segments (one lane walking all of K took 0.26 s for 4M
    elements).  Integers bit for bit (s8 widened to s32, s32 and u8 in their own wrapping types), floats within the
    bound of an accumulation in any order; batched once."""
    rng = np.random.default_rng(seed_of(M, N, K, ty, layout, "few outputs"))
    integer = ty in ("s8", "s32", "u8")
    a_shape = (M, K) if layout[0] == "n" else (K, M)
    b_shape = (K, N) if layout[1] == "n" else (N, K)
    if integer:
        lo, hi = (-127, 128) if ty != "u8" else (0, 256)
        a = rng.integers(lo, hi, size=a_shape).astype(T.numpy_dtype(T.normalize(ty)))
        b = rng.integers(lo, hi, size=b_shape).astype(T.numpy_dtype(T.normalize(ty)))
    else:
        a, b = rand_raw(rng, ty, a_shape, lo=-1, hi=1), rand_raw(rng, ty, b_shape, lo=-1, hi=1)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    kw = {"out_type": "s32"} if ty == "s8" else {}
    got, want = Nx.dot(ha, c1, hb, c2, **kw), Nx.dot(oa, c1, ob, c2, **kw)
    if integer:
        assert_bits_equal(got, want, f"dot {ty} {layout} {M}x{N}x{K}")
    else:
        eq = ("mk" if layout[0] == "n" else "km") + "," + ("kn" if layout[1] == "n" else "nk") + "->mn"
        check_float_dot(got, want, values(oa), values(ob), eq, K, f"dot {ty} {layout} {M}x{N}x{K}")


def test_few_outputs_over_a_long_contraction_batched(hip, oracle):
    rng = np.random.default_rng(77)
    a, b = rand_raw(rng, "f32", (3, 2, 6000), lo=-1, hi=1), rand_raw(rng, "f32", (3, 6000, 4), lo=-1, hi=1)
    ha, oa = both(a, "f32", hip, oracle)
    hb, ob = both(b, "f32", hip, oracle)
    got, want = Nx.dot(ha, [2], [0], hb, [1], [0]), Nx.dot(oa, [2], [0], ob, [1], [0])
    check_float_dot(got, want, values(oa), values(ob), "bmk,bkn->bmn", 6000, "batched few outputs")
    v = rng.integers(-100, 100, size=(1 << 20,)).astype(np.int32)
    hv, ov = both(v, "s32", hip, oracle)
    assert_bits_equal(Nx.dot(hv, hv), Nx.dot(ov, ov), "vector . vector s32")


@pytest.mark.parametrize("M,N,K", [(300, 10, 784), (1000, 1, 512), (65, 32, 256), (2000, 17, 128), (4099, 3, 1152)])
@pytest.mark.parametrize("ty", ["f32", "bf16", "f16", "s8"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_many_rows_against_a_few_columns(M, N, K, ty, layout, hip, oracle):
    """A layer with a few outputs ([60000, 784] . [784, 10]): tiles of 128 x 32, and a K that is not whole slabs
    with its partial slab walked in place.  int8 exact, floats within the accumulation bound,
    and every output in its own place (rows and columns off every tile edge)."""
    rng = np.random.default_rng(seed_of(M, N, K, ty, layout, "narrow"))
    if ty == "s8":
        a = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
        b = rng.integers(-127, 128, size=(K, N)).astype(np.int8)
    else:
        a, b = rand_raw(rng, ty, (M, K), lo=-1, hi=1), rand_raw(rng, ty, (K, N), lo=-1, hi=1)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    kw = {"out_type": "s32"} if ty == "s8" else {}
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2, **kw)
    assert got.shape == (M, N)
    rows = np.unique(np.concatenate([[0, 63, 64, min(127, M - 1), min(128, M - 1), M - 1], rng.integers(0, M, size=20)]))
    oa, ob = from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle)
    want = Nx.dot(oa, ob, **kw)
    got_rows = from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), "s32" if ty == "s8" else ty, oracle)
    if ty == "s8":
        assert_bits_equal(got_rows, want, f"narrow s8 {layout}")
        full = a.astype(np.int64) @ b.astype(np.int64)
        assert np.array_equal(hip.to_numpy(got).astype(np.int64), full)
    else:
        check_float_dot(got_rows, want, values(oa), values(ob), "mk,kn->mn", K, f"narrow {ty} {layout}")


def test_more_batch_items_than_a_grid_dimension_holds(hip, oracle):
    """100000 small matrices (a transform per point): the batch goes in runs of 65535 items.  Integer-valued f32, so
    every product and sum is exact and numpy's einsum is the answer bit for bit; a few items against the oracle."""
    rng = np.random.default_rng(31)
    a = rng.integers(-8, 9, size=(70001, 3, 3)).astype(np.float32)
    b = rng.integers(-8, 9, size=(70001, 3, 2)).astype(np.float32)
    got = Nx.dot(from_numpy(a, "f32", hip), [2], [0], from_numpy(b, "f32", hip), [1], [0])
    assert got.shape == (70001, 3, 2)
    assert np.array_equal(hip.to_numpy(got), np.einsum("bmk,bkn->bmn", a, b))
    pick = [0, 65534, 65535, 65536, 70000]
    want = Nx.dot(from_numpy(a[pick], "f32", oracle), [2], [0], from_numpy(b[pick], "f32", oracle), [1], [0])
    assert_bits_equal(from_numpy(hip.to_numpy(got)[pick], "f32", oracle), want, "batch of 70001")


@pytest.mark.parametrize("ty", ["f32", "bf16", "s32"])
def test_a_dot_product_per_batch_item(ty, hip, oracle):
    """[B, 1, K] . [B, K, 1]: one output per item, each a work-group of the reduction kernel."""
    rng = np.random.default_rng(seed_of(ty, "rowwise dot"))
    if ty == "s32":
        a, b = rng.integers(-100, 100, size=(3000, 1, 512)).astype(np.int32), rng.integers(-100, 100, size=(3000, 512, 1)).astype(np.int32)
    else:
        a, b = rand_raw(rng, ty, (3000, 1, 512), lo=-1, hi=1), rand_raw(rng, ty, (3000, 512, 1), lo=-1, hi=1)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    got, want = Nx.dot(ha, [2], [0], hb, [1], [0]), Nx.dot(oa, [2], [0], ob, [1], [0])
    if ty == "s32":
        assert_bits_equal(got, want, "row-wise dot s32")
    else:
        check_float_dot(got, want, values(oa), values(ob), "bmk,bkn->bmn", 512, f"row-wise dot {ty}")


def test_millions_of_rows_against_a_tiny_matrix(hip):
    """[2M, 3] . [3, 3] (points times a transform): K is not a multiple of 16 bytes, so the plain kernel runs, with
    131072 tiles of rows along the grid's first dimension.  Integer-valued f32: exact."""
    rng = np.random.default_rng(9)
    a = rng.integers(-8, 9, size=(2_000_003, 3)).astype(np.float32)
    b = rng.integers(-8, 9, size=(3, 3)).astype(np.float32)
    got = hip.to_numpy(Nx.dot(from_numpy(a, "f32", hip), from_numpy(b, "f32", hip)))
    assert np.array_equal(got, a @ b)


@pytest.mark.parametrize("ty", ["f64", "s32", "u8", "s64"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_plain_kernel_on_64_tiles(ty, layout, hip, oracle):
    """Types without a matrix-core path (f64, wide integers) on tiles of 64 x 64 with sixteen outputs per lane, from 512
    tiles on: every output is still accumulated over k in order, so integers are exact and f64 agrees with the oracle's
    sequential f64 sum bit for bit.  Shapes off the tile and K-step grids."""
    M, N, K = 1500, 1400, 37
    rng = np.random.default_rng(seed_of(ty, layout, "plain 64"))
    if ty == "f64":
        a, b = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    else:
        dt = T.numpy_dtype(T.normalize(ty))
        lo, hi = (0, 200) if ty == "u8" else (-1000, 1000)
        a, b = rng.integers(lo, hi, size=(M, K)).astype(dt), rng.integers(lo, hi, size=(K, N)).astype(dt)
    la = a if layout[0] == "n" else np.ascontiguousarray(a.T)
    lb = b if layout[1] == "n" else np.ascontiguousarray(b.T)
    c1 = [1] if layout[0] == "n" else [0]
    c2 = [0] if layout[1] == "n" else [1]
    got = Nx.dot(from_numpy(la, ty, hip), c1, from_numpy(lb, ty, hip), c2)
    rows = np.unique(np.concatenate([[0, 63, 64, M - 1], rng.integers(0, M, size=8)]))
    want = Nx.dot(from_numpy(np.ascontiguousarray(a[rows]), ty, oracle), from_numpy(b, ty, oracle))
    assert_bits_equal(from_numpy(np.ascontiguousarray(hip.to_numpy(got)[rows]), ty, oracle), want, f"plain 64 {ty} {layout}")
    if ty != "f64":
        wide = (a.astype(np.int64) @ b.astype(np.int64)).astype(T.numpy_dtype(T.normalize(ty)))
        assert np.array_equal(hip.to_numpy(got), wide)


@pytest.mark.parametrize("M,K,N", [(3, 3, 1), (4, 4, 4), (1, 7, 5), (8, 2, 8), (2, 64, 2)])
@pytest.mark.parametrize("ty", ["f32", "bf16", "s32", "f64"])
def test_many_small_matrices(M, K, N, ty, hip, oracle):
    """A batch of small matrices takes one lane per output over the whole batch; k in order, so the oracle's bits."""
    rng = np.random.default_rng(seed_of(M, K, N, ty, "small batched"))
    Bn = 777
    if ty == "s32":
        a, b = rng.integers(-99, 99, size=(Bn, M, K)).astype(np.int32), rng.integers(-99, 99, size=(Bn, K, N)).astype(np.int32)
    else:
        a, b = rand_raw(rng, ty, (Bn, M, K), lo=-2, hi=2), rand_raw(rng, ty, (Bn, K, N), lo=-2, hi=2)
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    assert_bits_equal(Nx.dot(ha, [2], [0], hb, [1], [0]), Nx.dot(oa, [2], [0], ob, [1], [0]), f"small batched {ty} {M}x{K}x{N}")
    # the other layouts: contract the first axis of the left operand, the last of the right
    at, bt = np.ascontiguousarray(a.transpose(0, 2, 1)), np.ascontiguousarray(b.transpose(0, 2, 1))
    hat, oat = both(at, ty, hip, oracle)
    hbt, obt = both(bt, ty, hip, oracle)
    assert_bits_equal(Nx.dot(hat, [1], [0], hbt, [2], [0]), Nx.dot(oat, [1], [0], obt, [2], [0]), f"small batched tt {ty}")


@pytest.mark.parametrize("S,R,K", [(1, 4096, 1024), (4, 1000, 300), (2, 257, 5000), (3, 70000, 256)])
@pytest.mark.parametrize("ty", ["f32", "f64", "s32"])
@pytest.mark.parametrize("side", ["vectors_left", "vectors_right"])
@pytest.mark.parametrize("small_layout", ["k_inner", "k_outer"])
def test_a_few_vectors_against_a_matrix(S, R, K, ty, side, small_layout, hip, oracle):
    """A few vectors against a matrix in f32 and wider types: with the matrix stored [N, K] (contiguous along k) the
    reduction kernel, a work-group per output; stored [K, N] the tiled kernels.  Integers exact, floats in the bound."""
    rng = np.random.default_rng(seed_of(S, R, K, ty, side, small_layout, "few vectors"))
    if ty == "s32":
        small, big = rng.integers(-99, 99, size=(S, K)).astype(np.int32), rng.integers(-99, 99, size=(K, R)).astype(np.int32)
    else:
        small, big = rand_raw(rng, ty, (S, K), lo=-1, hi=1), rand_raw(rng, ty, (K, R), lo=-1, hi=1)
    for big_layout in ("k_outer", "k_inner"):
        sm = small if small_layout == "k_inner" else np.ascontiguousarray(small.T)
        bg = big if big_layout == "k_outer" else np.ascontiguousarray(big.T)
        cs, cb = ([1] if small_layout == "k_inner" else [0]), ([0] if big_layout == "k_outer" else [1])
        hs, os_ = both(sm, ty, hip, oracle)
        hb, ob = both(bg, ty, hip, oracle)
        if side == "vectors_left":
            got, want, eq = Nx.dot(hs, cs, hb, cb), Nx.dot(os_, cs, ob, cb), "sk,kr->sr"
            a64, b64 = values(from_numpy(small, ty, oracle)), values(from_numpy(big, ty, oracle))
        else:
            got, want, eq = Nx.dot(hb, cb, hs, cs), Nx.dot(ob, cb, os_, cs), "kr,sk->rs"
            a64, b64 = values(from_numpy(big, ty, oracle)), values(from_numpy(small, ty, oracle))
        if ty == "s32":
            assert_bits_equal(got, want, f"few vectors s32 {side} {big_layout}")
        else:
            check_float_dot(got, want, a64, b64, eq, K, f"few vectors {ty} {side} {small_layout} {big_layout}")


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (256, 384, 512), (130, 70, 144), (1024, 1024, 256), (64, 2048, 1024), (33, 40, 16), (2000, 16, 4096)])
def test_f64_contraction_on_the_matrix_cores(M, N, K, layout, hip, oracle):
    """f64 operands whose K is a whole number of 128-byte slabs (16 elements) and whose result has 256 elements or more
    take the MFMA f64 path (`v_mfma_f64_16x16x4_f64`, f64 accumulators): within the accumulation bound of the oracle's
    sequential f64 sum, and exact where every partial sum is (small integers).  Other f64 shapes stay on the plain
    kernels, which add over k in order and so match the oracle bit for bit (test_plain_kernel_on_64_tiles)."""
    rng = np.random.default_rng(seed_of(M, N, K, layout, "f64 mfma"))
    a_shape = (M, K) if layout[0] == "n" else (K, M)
    b_shape = (K, N) if layout[1] == "n" else (N, K)
    c1, c2 = [1] if layout[0] == "n" else [0], [0] if layout[1] == "n" else [1]
    a, b = rng.standard_normal(a_shape), rng.standard_normal(b_shape)
    ha, oa = both(a, "f64", hip, oracle)
    hb, ob = both(b, "f64", hip, oracle)
    got, want = Nx.dot(ha, c1, hb, c2), Nx.dot(oa, c1, ob, c2)
    am = a if layout[0] == "n" else a.T
    bm = b if layout[1] == "n" else b.T
    check_float_dot(got, want, am, bm, "mk,kn->mn", K, f"f64 {M}x{N}x{K} {layout}")
    ai, bi = rng.integers(-50, 51, size=a_shape).astype(np.float64), rng.integers(-50, 51, size=b_shape).astype(np.float64)
    exact = (ai if layout[0] == "n" else ai.T) @ (bi if layout[1] == "n" else bi.T)
    res = hip.to_numpy(Nx.dot(from_numpy(ai, "f64", hip), c1, from_numpy(bi, "f64", hip), c2))
    assert np.array_equal(res, exact)
    # an f32 result from f64 operands: one rounding of the f64 sum
    res32 = hip.to_numpy(Nx.dot(from_numpy(ai, "f64", hip), c1, from_numpy(bi, "f64", hip), c2, out_type="f32"))
    assert np.array_equal(res32, exact.astype(np.float32))


@pytest.mark.parametrize("ty", ["f16", "bf16", "f32", "f64"])
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (5, 1, 7), (64, 1, 64), (3, 2, 4), (16, 16, 16), (33, 64, 40), (128, 128, 128), (1, 256, 1)])
def test_zero_products_leave_a_positive_zero(ty, m, k, n, hip, oracle):
    """The reference adds every product to a sum that starts at 0, so products that are all -0 (a negative factor
    times +0) give +0, with one term (K = 1) as with many; outputs whose terms cancel are +0 as well."""
    rng = np.random.default_rng(seed_of("zero products", ty, m, k, n))
    dtype = np.float32 if ty == "bf16" else T.numpy_dtype(T.normalize(ty))
    a = rng.choice(np.array([-1.0, -2.0, 1.0, 0.0, -0.0]), size=(m, k)).astype(dtype)
    b = rng.choice(np.array([0.0, -0.0, 0.0, 1.0, -1.0]), size=(k, n), p=[0.4, 0.3, 0.1, 0.1, 0.1]).astype(dtype)
    if ty == "bf16":
        a, b = [(np.asarray(v, np.float32).view(np.uint32) >> 16).astype(np.uint16) for v in (a, b)]
    ha, oa = both(a, ty, hip, oracle)
    hb, ob = both(b, ty, hip, oracle)
    assert_bits_equal(Nx.dot(ha, hb), Nx.dot(oa, ob), f"dot {ty} {m}x{k}x{n}")
    assert_bits_equal(Nx.dot(ha, [0], hb, [1]) if m == n else Nx.dot(hb, [0], ha, [1]),
                      Nx.dot(oa, [0], ob, [1]) if m == n else Nx.dot(ob, [0], oa, [1]), f"dot {ty} other axes")


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("lt,rt,M,N,K", [("f32", "f32", 80, 3, 1601), ("bf16", "bf16", 17, 33, 577), ("f16", "f16", 5, 61, 3333), ("f32", "f32", 16, 16, 640 + 33),
                                         ("f16", "f32", 20, 12, 1500), ("s32", "s32", 33, 40, 1333), ("f64", "f64", 20, 12, 1501), ("f32", "f32", 40, 9, 31)])
def test_few_outputs_over_a_long_k_are_cut_into_segments(lt, rt, M, N, K, layout, hip, oracle):
    """Plain kernels with K cut: integers exact; f64 operands are not cut and add in order of k (the oracle's bits); the others are f64
    sums in another order, K * 2^-53 of the magnitudes apart at most, rounded once to the result's type."""
    rng = np.random.default_rng(seed_of(lt, rt, M, N, K, layout, "segments"))
    arrays = [rng.integers(-999, 999, size=s).astype(np.int32) if t == "s32" else rand_raw(rng, t, s, lo=-1, hi=1)
              for t, s in ((lt, (M, K) if layout[0] == "n" else (K, M)), (rt, (K, N) if layout[1] == "n" else (N, K)))]
    (ha, oa), (hb, ob) = both(arrays[0], lt, hip, oracle), both(arrays[1], rt, hip, oracle)
    axes = [1] if layout[0] == "n" else [0], [0] if layout[1] == "n" else [1]
    got, want = Nx.dot(ha, axes[0], hb, axes[1]), Nx.dot(oa, axes[0], ob, axes[1])
    if lt in ("s32", "f64"):
        assert_bits_equal(got, want, f"{lt} {layout}")
        return
    a, b = values(oa) if layout[0] == "n" else values(oa).T, values(ob) if layout[1] == "n" else values(ob).T
    apart = np.abs(values(got) - values(want))
    assert (apart <= ULP[got.type] * np.abs(values(want)) + 2 * K * 2.0 ** -53 * (np.abs(a) @ np.abs(b))).all(), f"{lt} {layout}: {apart.max()}"


@pytest.mark.parametrize("ty", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(1, 256, 64), (8, 1000, 4096), (32, 136, 520), (17, 2048, 1096), (5, 11008, 256), (32, 128, 8200), (31, 392, 72)])
def test_few_rows_against_k_outer_weights_on_tiles_of_32(M, N, K, ty, hip):
    """Whole and partial slabs of K, K cut and whole, the edges of 32 rows and 128 columns: whole numbers, exact in any order."""
    rng = np.random.default_rng(seed_of(M, N, K, ty))
    a, b = rng.integers(-2, 3, size=(M, K)).astype(np.float32), rng.integers(-2, 3, size=(K, N)).astype(np.float32)

    def put(v):
        return from_numpy((v.view(np.uint32) >> 16).astype(np.uint16) if ty == "bf16" else v.astype(np.float16), ty, hip)
    exact = a.astype(np.float64) @ b
    got = values(Nx.dot(put(a), [1], put(b), [0]))
    want = (exact.astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32) if ty == "bf16" else exact.astype(np.float16)
    np.testing.assert_array_equal(got, want.astype(np.float64))


# f32 with an operand that is not K-inner: tiles of 64 x 128 and 128 x 128 on eight waves up to one or two work-groups to a CU and
# on four beyond, one slab, a partial slab, K cut
@pytest.mark.parametrize("layout", ["nn", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(64, 256, 32), (68, 132, 36), (60, 384, 68), (1000, 132, 64), (2044, 1028, 40), (4100, 1024, 36), (4096, 2052, 100),
                                   (2048, 2048, 96), (300, 1000, 900), (1024, 1024, 260), (132, 260, 4100)])
def test_f32_tiles_on_four_and_eight_waves(M, N, K, layout, hip):
    """Whole numbers whose sums are exact in f32 in any order, so every output is the same number on any kernel."""
    rng = np.random.default_rng(seed_of(M, N, K, layout))
    a, b = rng.integers(-3, 4, size=(M, K)).astype(np.float32), rng.integers(-3, 4, size=(K, N)).astype(np.float32)
    l, lc = (a, [1]) if layout[0] == "n" else (np.ascontiguousarray(a.T), [0])
    r, rc = (b, [0]) if layout[1] == "n" else (np.ascontiguousarray(b.T), [1])
    got = values(Nx.dot(from_numpy(l, "f32", hip), lc, from_numpy(r, "f32", hip), rc))
    np.testing.assert_array_equal(got, a.astype(np.float64) @ b.astype(np.float64))


# Tiles and ranges by the cost model: 64 x 64 and 64 x 128 on the two-group kernel, 32 x 128 against K-outer weights, one slab and odd
# numbers of them, K cut with ranges of unequal length, the batch beside them
@pytest.mark.parametrize("ty", ["bf16", "f16", "s8"])
@pytest.mark.parametrize("right", ["n", "t"])
@pytest.mark.parametrize("batch,M,N,K", [(1, 500, 500, 500), (1, 65, 129, 64), (1, 1000, 2000, 504), (1, 100, 300, 8000), (1, 256, 1025, 4160), (3, 200, 328, 1336),
                                         (1, 129, 1000, 128), (1, 66, 4096, 11016), (1, 260, 520, 2240)])
def test_tiles_of_small_and_middling_contractions(ty, right, batch, M, N, K, hip):
    """Whole numbers whose sums are exact in f32 in any order, so every output is the same number on any kernel."""
    rng = np.random.default_rng(seed_of(ty, right, batch, M, N, K))
    a, b = rng.integers(-3, 4, size=(batch, M, K)), rng.integers(-3, 4, size=(batch, K, N))
    lb = b if right == "n" else np.ascontiguousarray(b.transpose(0, 2, 1))
    got = Nx.dot(from_numpy(HELD[ty](a), ty, hip), [2], [0], from_numpy(HELD[ty](lb), ty, hip), [1 if right == "n" else 2], [0], out_type="s32" if ty == "s8" else "f32")
    assert np.array_equal(hip.to_numpy(got).astype(np.float64), a.astype(np.float64) @ b.astype(np.float64))


@pytest.mark.parametrize("M,N,K,contract", [(48, 384, 9568, 1), (256, 1025, 8192, 0), (130, 257, 9999, 1), (64, 4098, 11008, 1)])
@pytest.mark.parametrize("mode", ["column", "row", "one"])
def test_scaled_int8_sums_of_cut_contractions(M, N, K, contract, mode, hip):
    """K cut into ranges: their whole sums, converted and scaled once each, as numpy gives them in f32."""
    from nx_amd._lib import SCALE_ONE, SCALE_PER_COLUMN, SCALE_PER_ROW
    rng = np.random.default_rng(seed_of(M, N, K, contract, mode, "cut and scaled"))
    x, w = rng.integers(-127, 128, size=(M, K)).astype(np.int8), rng.integers(-127, 128, size=(N, K)).astype(np.int8)
    s = rng.uniform(1e-3, 1e-2, size={"column": N, "row": M, "one": 1}[mode]).astype(np.float32)
    sums = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.float32)  # exact below 2^53, rounded once
    want = sums * (s[None, :] if mode == "column" else s[:, None] if mode == "row" else s)
    held = w if contract else np.ascontiguousarray(w.T)
    sc = from_numpy(s, "f32", hip)
    out = hip.dot_scaled(sc.with_(data=None, shape=(M, N)), from_numpy(x, "s8", hip), [1], [], from_numpy(held, "s8", hip), [contract], [], sc,
                         {"column": SCALE_PER_COLUMN, "row": SCALE_PER_ROW, "one": SCALE_ONE}[mode], any_k=True)
    np.testing.assert_array_equal(hip.to_numpy(out), want)
