"""Products at the edges of their kernels' tiles, k-tiles and slices, against
float64: integer operands small enough that every F32 sum is exact, so any
order gives the same bits, or random ones within a derived bound.
"""
import numpy as np
import pytest

import miburn
from miburn import bf16_bits, bf16_to_f32

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(41)


def _ints(shape, lo=-2, hi=3):
    return RNG.integers(lo, hi, shape).astype(np.float32)


@pytest.mark.parametrize("m,n,k", [(640, 320, 4000), (64, 64, 2080), (128, 192, 1056)])
def test_bf16_split_k_of_a_half_k_tile(engine, m, n, k):
    """k a multiple of 32 and not of the 64-wide k-tile, split over k: the last
    slice ends inside its k-tile and reads nothing past it."""
    a, b = _ints((m, k)), _ints((k, n))
    ia, ib = engine.upload_bf16(bf16_bits(a)), engine.upload_bf16(bf16_bits(b))
    o = engine.matmul_dram(ia, False, ib, False)
    got = engine.download(o)
    for t in (ia, ib, o):
        engine.free(t)
    assert np.array_equal(got, (a.astype(np.float64) @ b).astype(np.float32))


# Shapes that reach the direct kernel through packed operands: each edge of
# its 256 x 256 and 128 x 128 tiles, k off the k-tile, both orientations,
# in-place operands whose rows end mid-block or mid-tile, BF16 results.
@pytest.mark.parametrize("m,n,k,ta,tb,out", [
    (1000, 1000, 1000, False, False, "f32"),   # k % 32, packed both
    (1001, 1023, 512, False, True, "f32"),     # in place, rows off the DMA's blocks
    (1001, 1016, 512, False, False, "f32"),    # in place, columns in eights
    (777, 2049, 257, False, False, "bf16"),    # odd pitch, one column past a tile
    (513, 1025, 640, True, False, "f32"),      # transposed A
    (3585, 3841, 96, True, True, "f32"),       # 256-row tiles, one past the last
    (1501, 3065, 512, False, True, "f32"),     # 192 x 128 tiles
    (1501, 3064, 500, False, False, "bf16"),
    (3001, 2500, 512, False, True, "f32"),     # 256 x 128 tiles
    (3001, 2497, 500, False, False, "f32"),
])
def test_bf16_any_shape(engine, m, n, k, ta, tb, out):
    a, b = _ints((k, m) if ta else (m, k)), _ints((n, k) if tb else (k, n))
    ia, ib = engine.upload_bf16(bf16_bits(a)), engine.upload_bf16(bf16_bits(b))
    o = engine.matmul_dram(ia, ta, ib, tb, miburn.BF16 if out == "bf16" else miburn.F32)
    got = engine.download(o)
    for t in (ia, ib, o):
        engine.free(t)
    want = ((a.T if ta else a) @ (b.T if tb else b)).astype(np.float32)  # exact: |sums| < 2^24
    if out == "bf16":
        got, want = got, bf16_bits(want)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("bcast", ["none", "a", "b"])
def test_bf16_any_shape_batched(engine, bcast):
    bt, m, n, k = 6, 500, 490, 250
    a, b = _ints((1 if bcast == "a" else bt, m, k)), _ints((1 if bcast == "b" else bt, k, n))
    ia = engine.upload_bf16(bf16_bits(a.reshape(-1, k)))
    ib = engine.upload_bf16(bf16_bits(b.reshape(-1, n)))
    o = engine.matmul_dram_batched(ia, False, ib, False, bt, m, k, n)
    got = engine.download(o).reshape(bt, m, n)
    for t in (ia, ib, o):
        engine.free(t)
    assert np.array_equal(got, np.matmul(a, b))


@pytest.mark.parametrize("ea,eb,m,n,k,ta,tb", [
    ("f32", "f32", 2051, 2049, 2050, False, False),
    ("f32", "f32", 2051, 2049, 2050, True, True),
    ("bf16", "f32", 2051, 2049, 2050, False, True),
    ("f32", "bf16", 1501, 2051, 800, False, True),
    ("f32", "bf16", 1501, 2050, 801, True, False),
])
def test_f32_any_shape_fast(engine, ea, eb, m, n, k, ta, tb):
    """The fast mode's parts: error per product within 3 * 2^-18 |a||b| and the
    F32 accumulation's 2 K * 2^-24, each against sum |a||b|."""
    a, b = (RNG.standard_normal(s).astype(np.float32) for s in ((k, m) if ta else (m, k), (n, k) if tb else (k, n)))
    up = {"f32": engine.upload, "bf16": lambda x: engine.upload_bf16(bf16_bits(x))}
    av, bv = (x if e == "f32" else bf16_to_f32(bf16_bits(x)) for x, e in ((a, ea), (b, eb)))
    ia, ib = up[ea](a), up[eb](b)
    o = engine.matmul_dram(ia, ta, ib, tb)
    got = engine.download(o)
    for t in (ia, ib, o):
        engine.free(t)
    av, bv = (av.T if ta else av).astype(np.float64), (bv.T if tb else bv).astype(np.float64)
    bound = (3 * 2.0 ** -18 + 2 * k * 2.0 ** -24) * (np.abs(av) @ np.abs(bv))
    assert np.all(np.abs(got - av @ bv) <= bound)


def test_f32_any_shape_bias_residual(engine):
    m, n, k = 1501, 2051, 801
    x, w = _ints((m, k)), _ints((n, k))
    bias, res = _ints((1, n)), _ints((m, n))
    ids = [engine.upload(x), engine.upload_bf16(bf16_bits(w)), engine.upload(bias), engine.upload(res)]
    o = engine.linear(ids[0], ids[1], True, ids[2], ids[3])
    got = engine.download(o)
    for t in ids + [o]:
        engine.free(t)
    assert np.array_equal(got, res + (x @ w.T + bias))


# F32 products at F32 precision: each tile (64 x 64, 64 x 128, 128 x 128),
# whole and with edges, each DMA width, k-tile remainders, one k-tile, slices.
F32_SHAPES = [(64, 64, 32), (64, 64, 8), (65, 67, 33), (1, 1, 1), (130, 66, 20), (128, 192, 96), (512, 512, 512),
              (2048, 768, 256), (2050, 772, 260), (2049, 771, 259), (2048, 2048, 64), (2052, 2044, 68),
              (257, 129, 2047), (1500, 1500, 300)]


def _f32_product(engine, a, ta, b, tb):
    ia, ib = engine.upload(a), engine.upload(b)
    o = engine.matmul_dram(ia, ta, ib, tb)
    got = engine.download(o)
    for t in (ia, ib, o):
        engine.free(t)
    return got


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n,k", F32_SHAPES)
def test_f32_precise_product(engine, m, n, k, ta, tb):
    """Against float64 within an F32 sum's bound, k + 4 roundings of 2^-24 of
    sum |a||b| (the parts left out of a product: 2^-24 of it)."""
    a, b = (RNG.standard_normal(s).astype(np.float32) for s in ((k, m) if ta else (m, k), (n, k) if tb else (k, n)))
    got = _f32_product(engine, a, ta, b, tb)
    av, bv = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
    assert np.all(np.abs(got - av @ bv) <= (k + 4) * 2.0 ** -24 * (np.abs(av) @ np.abs(bv)))


@pytest.mark.parametrize("m,n,k", [(64, 64, 40), (1024, 2048, 256), (2048, 2048, 64)])
def test_f32_non_finite_operands(engine, m, n, k):
    """An infinity, a NaN, a value next to the largest and zeros against them
    give what F32 arithmetic gives, also where parts are multiplied."""
    a, b = RNG.standard_normal((m, k)).astype(np.float32), RNG.standard_normal((k, n)).astype(np.float32)
    a[3, 5], a[7, 1], a[9, 2], a[m - 1, k - 1] = np.inf, np.nan, np.float32(3.4028e38), -np.inf
    b[5, 4] = b[2, 11] = 0.0
    b[2, :8] = 0.25
    got = _f32_product(engine, a, False, b, False)
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        want = np.where(np.abs(want) > np.finfo(np.float32).max, np.copysign(np.inf, want), want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32)) and not np.isinf(got[~inf]).any()
    row9 = np.isfinite(want[9])
    assert np.allclose(got[9][row9], want[9][row9], rtol=1e-6)


def test_f32_sum_has_no_bias(engine):
    """A sum over the rows of a product of parts: its error is the rounding
    errors' sum, not their number times a bias (2e-8 of a value each)."""
    m, n, k = 2048, 2048, 512
    a, b = RNG.standard_normal((m, k)).astype(np.float32), RNG.standard_normal((k, n)).astype(np.float32)
    d = _f32_product(engine, a, False, b, False) - a.astype(np.float64) @ b.astype(np.float64)
    sd = d.std()
    assert abs(d.mean()) < 6 * sd / np.sqrt(m * n)                       # independent errors' mean
    assert np.abs(d.mean(axis=0)).max() < 7 * sd / np.sqrt(m)            # and each column's


# ------------------------------------------------------ rows of any width
WIDE_ROWS = [(3, 1025), (5, 2048), (7, 2049), (300, 4095), (2, 4097), (9, 8001), (4, 8192)]


@pytest.mark.parametrize("rows,cols", WIDE_ROWS)
def test_wide_row_norms(engine, rows, cols):
    """RMSNorm and LayerNorm with a block a row, against float64: rel 1e-5."""
    x = (RNG.standard_normal((rows, cols)) + 0.5).astype(np.float32)
    g, b = RNG.standard_normal((1, cols)).astype(np.float32), RNG.standard_normal((1, cols)).astype(np.float32)
    ids = [engine.upload(t) for t in (x, g, b)]
    xd = x.astype(np.float64)
    rms = xd / np.sqrt((xd * xd).mean(1, keepdims=True) + 1e-5)
    c = xd - xd.mean(1, keepdims=True)
    ln = c / np.sqrt((c * c).mean(1, keepdims=True) + 1e-5)
    for o, want in ((engine.rms_norm(ids[0], ids[1]), rms * g), (engine.rms_norm(ids[0]), rms),
                    (engine.layer_norm(ids[0], ids[1], ids[2]), ln * g + b), (engine.layer_norm(ids[0]), ln)):
        got = engine.download(o)
        engine.free(o)
        assert np.abs(got - want).max() <= 1e-5 * max(1.0, np.abs(want).max())
    for t in ids:
        engine.free(t)


@pytest.mark.parametrize("rows,cols", [(1, 512), (3, 515), (300, 2049), (5, 8001), (4097, 1023), (256, 1), (256, 33),
                                       (64, 128), (257, 40), (7, 100000)])
def test_row_and_column_folds(engine, rows, cols):
    """Sums, maxima, minima and means over either axis, and a NaN in them."""
    x = RNG.standard_normal((rows, cols)).astype(np.float32)
    ix = engine.upload(x)
    for axis, ax in ((miburn.AXIS_COLS, 1), (miburn.AXIS_ROWS, 0)):
        n = x.shape[ax]
        for op, f in ((miburn.R_SUM, np.sum), (miburn.R_MEAN, np.mean), (miburn.R_MAX, np.max), (miburn.R_MIN, np.min)):
            o = engine.reduce(ix, op, axis)
            got = engine.download(o).reshape(-1)
            engine.free(o)
            want = f(x.astype(np.float64), axis=ax)
            if op in (miburn.R_MAX, miburn.R_MIN):
                assert np.array_equal(got, want.astype(np.float32))
            else:  # n roundings of 2^-24 of sum |x|
                bound = n * 2.0 ** -24 * np.abs(x).astype(np.float64).sum(ax) / (n if op == miburn.R_MEAN else 1)
                assert np.all(np.abs(got - want) <= bound + 1e-30)
    engine.free(ix)
    x[0, cols // 2] = np.nan
    ix = engine.upload(x)
    for op in (miburn.R_SUM, miburn.R_MAX, miburn.R_MIN):
        o = engine.reduce(ix, op, miburn.AXIS_COLS)
        got = engine.download(o).reshape(-1)
        engine.free(o)
        assert np.isnan(got[0]) and not np.isnan(got[1:]).any()
    engine.free(ix)


@pytest.mark.parametrize("n", [1, 64, 2048, 2049])
def test_whole_folds(engine, n):
    x = RNG.standard_normal((1, n)).astype(np.float32)
    ix = engine.upload(x)
    for op, f in ((miburn.R_SUM, np.sum), (miburn.R_MEAN, np.mean), (miburn.R_MAX, np.max)):
        o = engine.reduce_all(ix, op)
        got = float(engine.download(o)[0, 0])
        engine.free(o)
        assert abs(got - f(x.astype(np.float64))) <= n * 2.0 ** -24 * max(1e-3, np.abs(x).sum() / (n if f is np.mean else 1))
    engine.free(ix)


# Products over a long k with few tiles are summed in slices: the error of one
# F32 chain of n = k / 16 matrix-core steps is a random walk of roundings of
# partial sums that grow as sqrt(i), 0.4 * 2^-24 * sqrt(n / 2) of the result,
# and slices stay below it (1.0e-7 at the first; one chain reaches 2.2e-7).
@pytest.mark.parametrize("m,n,k,ta,tb", [
    (1656, 372, 1415, False, True),
    (777, 777, 3001, False, False),
    (300, 300, 3001, False, True),
])
def test_bf16_long_k_keeps_its_slices(engine, m, n, k, ta, tb):
    rng = np.random.default_rng(k)
    a = bf16_to_f32(bf16_bits(rng.standard_normal((k, m) if ta else (m, k), dtype=np.float32)))
    b = bf16_to_f32(bf16_bits(rng.standard_normal((n, k) if tb else (k, n), dtype=np.float32)))
    ia, ib = engine.upload_bf16(bf16_bits(a)), engine.upload_bf16(bf16_bits(b))
    o = engine.matmul_dram(ia, ta, ib, tb, miburn.F32)
    got = engine.download(o).astype(np.float64).reshape(m, n)
    for i in (ia, ib, o):
        engine.free(i)
    want = (a.T if ta else a).astype(np.float64) @ (b.T if tb else b).astype(np.float64)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < 0.4 * 2.0 ** -24 * np.sqrt(k / 32)


@pytest.mark.parametrize("m,n", [(4096, 4096), (2047, 2049)])
@pytest.mark.parametrize("k", [1, 2, 7, 8, 9, 33])
def test_f32_short_k_is_f32_arithmetic(engine, m, n, k):
    """Sums of few products over results large enough for any tile: an outer
    product is one rounding of each product, 2^-24 of it, and k products at
    most k of sum |a||b| (each product's and each sum's but the first)."""
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    got = _f32_product(engine, a, False, b, False)
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.all(np.abs(got - want) <= k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b)) * (1 + 2.0 ** -20))


# 64 x 128 and 128 x 128 tiles, whole, with edges and by 4-byte DMA; 64 x 128 in
# slices, the last of them one k-tile of 4.
@pytest.mark.parametrize("m,n,k", [(2048, 768, 256), (2048, 2048, 512), (1500, 1500, 300), (2049, 771, 259),
                                   (256, 768, 2308)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
@pytest.mark.parametrize("small", ["a", "b", "one column", "subnormal"])
def test_f32_small_operands(engine, m, n, k, ta, tb, small):
    """Values whose last bits lie below BF16's least subnormal (2^-133), down to
    F32's own subnormals, against ones that bring their products to ordinary
    size: an F32 sum's bound, as for any other values."""
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    if small == "one column":  # of A, and its row of B far above the rest
        a[:, 5] = np.ldexp(a[:, 5], -124)
        b[5] = np.ldexp(b[5], 124)
        b[:5], b[6:] = b[:5] * 2.0 ** -30, b[6:] * 2.0 ** -30
    elif small == "b":
        a, b = np.ldexp(a, 100), np.ldexp(b, -124)
    else:
        a, b = np.ldexp(a, -124 if small == "a" else -132), np.ldexp(b, 100)
    a, b = a.astype(np.float32), b.astype(np.float32)
    got = _f32_product(engine, a.T.copy() if ta else a, ta, b.T.copy() if tb else b, tb)
    av, bv = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(got - av @ bv) <= (k + 4) * 2.0 ** -24 * (np.abs(av) @ np.abs(bv)))


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 512), (1500, 1500, 300), (2048, 768, 256), (2049, 771, 259)])
def test_f32_non_finite_operands_on_every_parts_tile(engine, m, n, k):
    """An infinity, a NaN and a value next to the largest on 128 x 128 tiles
    whole and with edges, 64 x 128 ones, and by 4-byte DMA; the finite results
    within an F32 sum's bound."""
    rng = np.random.default_rng(n)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a[3, 5], a[7, 1], a[9, 2], a[m - 1, k - 1] = np.inf, np.nan, np.float32(3.4028e38), -np.inf
    b[5, 4] = b[2, 11] = 0.0
    b[2] *= 0.125
    got = _f32_product(engine, a, False, b, False)
    with np.errstate(all="ignore"):
        want, mag = a.astype(np.float64) @ b, np.abs(a).astype(np.float64) @ np.abs(b)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf, fin = np.isinf(want), np.isfinite(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32))
    assert np.all(np.abs(got[fin] - want[fin]) <= (k + 4) * 2.0 ** -24 * mag[fin])


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 512), (256, 768, 2308)])  # 128 x 128 whole; a slice of one k-tile
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_f32_product_on_parts_tiles(engine, m, n, k, ta, tb):
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    got = _f32_product(engine, a.T.copy() if ta else a, ta, b.T.copy() if tb else b, tb)
    av, bv = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(got - av @ bv) <= (k + 4) * 2.0 ** -24 * (np.abs(av) @ np.abs(bv)))
    again = _f32_product(engine, a.T.copy() if ta else a, ta, b.T.copy() if tb else b, tb)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(32, 2064), (288, 4096), (512, 3008), (544, 8192), (3, 2049), (5, 4098), (7, 2052)])
def test_wide_rms_norm_forms_are_its_f32_result(engine, rows, cols):
    """BF16, parts and tiled results of a block-a-row RMSNorm: the F32 result
    rounded, its heads and remainders, and the same in tiles, bit for bit."""
    rng = np.random.default_rng(cols)
    x, g = (engine.upload(rng.standard_normal(d).astype(np.float32)) for d in ((rows, cols), (1, cols)))
    y = engine.rms_norm(x, g)
    yv = engine.download(y)
    hi = bf16_bits(yv)
    lo = bf16_bits(yv - bf16_to_f32(hi))
    ids = [x, g, y]

    def form(f):
        ids.append(engine.rms_norm(x, g, 1e-5, f))
        return engine.download(ids[-1])
    assert np.array_equal(form(miburn.BF16), hi)
    assert np.array_equal(form(miburn.BF16_PARTS), np.concatenate([hi, lo], 1))
    if rows % 32 == 0 and cols % 16 == 0:
        for f in (miburn.TILES_BF16, miburn.TILES_PARTS):
            ids.append(engine.tile(y, f))
            assert np.array_equal(form(f).reshape(-1), engine.download(ids[-2]).reshape(-1))
    for t in ids:
        engine.free(t)


# ----------------------------------------------- more rows than one launch
# A launch holds fewer than 2^32 threads: rows past those that a block each
# fills it with.
@pytest.fixture
def own_engine():
    with miburn.Engine(0) as eng:  # its tens of GB are given back with it
        yield eng


def test_reduce_of_2_24_rows(own_engine):
    rows, cols = (1 << 24) + 3, 515
    x = own_engine.fill(rows, cols, miburn.F32, int(np.float32(1.0).view(np.uint32)))
    own_engine.assign_block(x, own_engine.upload(_ints((2, cols))), rows - 2, 0)
    tail = own_engine.download(own_engine.copy_strided(x, 2, cols, (rows - 2) * cols, cols, 1))
    got = own_engine.download(own_engine.reduce(x, miburn.R_SUM, miburn.AXIS_COLS)).reshape(-1)
    assert np.all(got[:-2] == cols) and np.array_equal(got[-2:], tail.sum(1))


@pytest.mark.parametrize("op,rows,cols", [("rms", (1 << 22) + 32, 4112), ("layer", (1 << 24) + 1, 1026)])
def test_norms_of_many_wide_rows(own_engine, op, rows, cols):
    x = own_engine.fill(rows, cols, miburn.F32, int(np.float32(2.0).view(np.uint32)))
    last = RNG.standard_normal((1, cols)).astype(np.float32)
    own_engine.assign_block(x, own_engine.upload(last), rows - 1, 0)
    if op == "rms":
        y, want = own_engine.rms_norm(x, 0, 0.0, miburn.BF16), last / np.sqrt((last.astype(np.float64) ** 2).mean())
    else:
        y, want = own_engine.layer_norm(x), (last - last.mean()) / np.sqrt(last.astype(np.float64).var() + 1e-5)
    got = own_engine.download(own_engine.copy_strided(y, 3, cols, (rows - 3) * cols, cols, 1))
    got = bf16_to_f32(got) if op == "rms" else got
    assert np.array_equal(got[:2], np.full((2, cols), 1.0 if op == "rms" else 0.0))
    assert np.abs(got[2] - want).max() <= (2.0 ** -8 if op == "rms" else 1e-5) * np.abs(want).max()
