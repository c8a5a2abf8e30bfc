"""The split GEMM (gemm_split.hpp): f32 products as six products of bf16 pieces.

plan.TILES has products for every tile of its planner, ragged and whole (that
they reach it is checked on the CPU); the other shapes add what lies about it:
one row or column past a tile, k remainders under and over a step, misaligned
operands (odd leading dimensions, pointers off 16 bytes), K slices, and small
products that the short GEMM kernel takes.

Bars: bit-exact where every product and partial sum is an integer below 2^24
(one operand of up to 18 bits, so all three of its pieces carry bits); against
f64, |C - C64| <= R * 2^-24 * (|A||B|) element by element, R as follows. A
bf16 instruction adds its 16 products in two halves of 8: in each, bits of the
products below 2^-24 of the largest are dropped (at most 7 such units), then the
accumulator is rounded to nearest (measured on the instruction with sums that
tell). Over a reduction the drops come to at most 7 units of |A||B|, the three
products of pieces left out to 1 and adding the two accumulators to 1. The
roundings are one unit of the sum so far: 6 K / 8 with one accumulator (256x256
tiles), else K / 8 of the large one and 5 K / 8 of one that holds 2^-7 of
|A||B|. K slices add one each. The f32 kernels round every product's sum: K.
"""
import numpy as np
import pytest

import plan
from kat import int_matrix

pytestmark = pytest.mark.gpu

NN, NT, TN = 0, 1, 2

TILES = [shape for shape, _ in plan.TILES]
SHAPES = [  # rows, cols, inner
    (33, 33, 32), (64, 64, 64), (65, 63, 33), (129, 200, 47),  # the short GEMM kernel
    (1000, 1333, 65), (1500, 1500, 100), (2048, 2048, 96), (2049, 2047, 80),  # 64x64 tiles
    (4096, 256, 130), (4100, 4090, 40),
    (4096, 4096, 48),                    # whole 256x256 tiles
    (64, 576, 5000), (70, 130, 4099), (520, 260, 2100),  # K slices
]
ALL = SHAPES + [t for t in TILES if t not in SHAPES]
IDS = lambda s: "x".join(map(str, s))


def roundings(layout, rows, cols, inner):
    """R of the bars."""
    cd = lambda a, b: -(-a // b)
    answer = plan.ask(("gemm", plan.LAYOUTS[layout], rows, cols, inner, 1, 0, 1, plan.CUS))[0]
    short = 2 * cd(rows, 64) * cd(cols, 64) <= plan.CUS and cd(rows, 16) * cd(cols, 16) <= 4 * plan.CUS \
        and inner <= 2048
    if short or answer == "f32":
        return inner + 8
    tile, slices, _ = answer.split()
    halves = cd(inner, 8)
    return 9 + (6 * halves if tile == "256x256x16" else halves * (1 + 5 / 128 * 1.02)) + \
        (int(slices) if slices != "1" else 0)


def operands(layout, rows, cols, inner, make_a, make_b):
    a = make_a((rows, inner) if layout != TN else (inner, rows))
    b = make_b((inner, cols) if layout != NT else (cols, inner))
    return a, b


def logical(layout, a, b):
    return (a.T if layout == TN else a).astype(np.float64), \
           (b.T if layout == NT else b).astype(np.float64)


def upload(hip, x, offset):
    """x on the device, `offset` floats past a 16-byte boundary."""
    buf = hip.DeviceBuffer.from_host(np.concatenate([np.zeros(offset, np.float32), x.ravel()]))
    return buf, buf.ptr + 4 * offset


def gemm(hip, layout, a, b, rows, cols, inner, offset=0, **kw):
    keep_a, pa = upload(hip, a, offset)
    keep_b, pb = upload(hip, b, offset)
    c = hip.DeviceBuffer.from_host(kw.pop("c0", np.full((rows, cols), np.nan, np.float32)))
    hip.gemm(layout, c, pa, pb, rows, cols, inner, **kw)
    return c.to_host((rows, cols))


@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", ALL, ids=IDS)
def test_exact_integers_all_pieces(hip, layout, shape):
    rows, cols, inner = shape
    rng = np.random.default_rng(rows + 3 * cols + 7 * inner + layout)
    bits = min(18, 23 - int(np.ceil(np.log2(inner))))  # sums of inner of them stay below 2^24
    wide = lambda s: int_matrix(rng, s, -2 ** bits + 1, 2 ** bits - 1)
    sign = lambda s: int_matrix(rng, s, -1, 1)
    for offset, (ma, mb) in enumerate([(wide, sign), (sign, wide)]):
        a, b = operands(layout, rows, cols, inner, ma, mb)
        A, B = logical(layout, a, b)
        got = gemm(hip, layout, a, b, rows, cols, inner, offset=offset)
        assert np.array_equal(got.astype(np.float64), A @ B)


@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(33, 33, 32), (129, 200, 47), (1000, 1333, 777),
                                   (2049, 2047, 300), (4096, 256, 1024), (64, 576, 20001)] + TILES,
                         ids=IDS)
def test_f64_error(hip, layout, shape):
    rows, cols, inner = shape
    rng = np.random.default_rng(rows + cols + inner + layout)
    # magnitudes over nine decades
    make = lambda s: (rng.standard_normal(s) * 10.0 ** rng.integers(-6, 4, s)).astype(np.float32)
    a, b = operands(layout, rows, cols, inner, make, make)
    A, B = logical(layout, a, b)
    sample = np.unique(np.linspace(0, rows - 1, 97).astype(int))
    got = gemm(hip, layout, a, b, rows, cols, inner)[sample]
    bound = roundings(layout, *shape) * 2.0 ** -24 * (np.abs(A[sample]) @ np.abs(B))
    assert np.all(np.abs(got - A[sample] @ B) <= bound)


@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(129, 200, 70), (1500, 1500, 100), (4096, 256, 130)] + TILES, ids=IDS)
def test_epilogues_exact(hip, layout, shape):
    rows, cols, inner = shape
    rng = np.random.default_rng(rows + layout)
    small = lambda s: int_matrix(rng, s, -8, 8)
    a, b = operands(layout, rows, cols, inner, small, small)
    A, B = logical(layout, a, b)
    c0, bc, br = small((rows, cols)), small(cols), small(rows)
    got = gemm(hip, layout, a, b, rows, cols, inner, c0=c0, beta=2.0, bias=hip.DeviceBuffer.from_host(bc),
               epilogue=hip.EPI_BIAS_COL | hip.EPI_RELU)
    assert np.array_equal(got, np.maximum(A @ B + bc, 0) + 2 * c0)
    got = gemm(hip, layout, a, b, rows, cols, inner, bias=hip.DeviceBuffer.from_host(br),
               epilogue=hip.EPI_BIAS_ROW)
    assert np.array_equal(got, A @ B + br[:, None])


@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(129, 200, 70), (1500, 1500, 100), (64, 576, 5000),
                                   (4096, 256, 130)] + TILES, ids=IDS)
def test_infinities_nan_and_overflow(hip, layout, shape):
    """The results that are not finite are those of f32 multiplication and
    addition, and every other one is exact."""
    rows, cols, inner = shape
    rng = np.random.default_rng(7 * rows + layout)
    small = lambda s: int_matrix(rng, s, 1, 8)  # no zeros: inf * 0 only where put
    a, b = operands(layout, rows, cols, inner, small, small)
    A, B = (a.T if layout == TN else a), (b.T if layout == NT else b)  # views
    A[3, 5] = np.inf
    A[rows - 1, inner - 1] = -np.inf
    A[7, 2] = np.nan
    B[4, cols - 2] = np.inf
    B[5, 1] = 0.0                          # inf * 0
    A[11, 0] = np.float32(3.4028235e38)    # rounds past bf16's range, finite
    B[0, :] = 0.5
    got = gemm(hip, layout, a, b, rows, cols, inner)
    with np.errstate(all="ignore"):
        want = np.zeros((rows, cols), np.float64)
        fa, fb = np.where(np.isfinite(A), A, 0).astype(np.float64), \
            np.where(np.isfinite(B), B, 0).astype(np.float64)
        want = fa @ fb
        for r, k in ((3, 5), (rows - 1, inner - 1), (7, 2)):
            want[r] += np.float64(A[r, k]) * B[k].astype(np.float64)
        want[:, cols - 2] += A[:, 4].astype(np.float64) * np.inf
    big = np.zeros((rows, cols), bool)
    big[11] = True
    finite = np.isfinite(want) & ~big
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    assert np.array_equal(got[finite].astype(np.float64), want[finite])
    row = np.isfinite(want[11])
    assert np.allclose(got[11][row], want[11][row], rtol=2.0 ** -22)


@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(129, 200, 70), (1500, 1500, 100), (4096, 256, 130)] + TILES, ids=IDS)
def test_tiny_magnitudes(hip, layout, shape):
    """Operands whose third piece lies under bf16's smallest denormal (2^-133)
    lose no precision: the results are those of f32 products."""
    rows, cols, inner = shape
    rng = np.random.default_rng(5 * rows + layout)
    tiny = lambda s: np.ldexp(rng.standard_normal(s), -118).astype(np.float32)
    unit = lambda s: np.ldexp(rng.standard_normal(s), 20).astype(np.float32)
    a, b = operands(layout, rows, cols, inner, tiny, unit)
    A, B = logical(layout, a, b)
    sample = np.unique(np.linspace(0, rows - 1, 97).astype(int))
    got = gemm(hip, layout, a, b, rows, cols, inner)[sample]
    bound = (inner + 8) * 2.0 ** -24 * (np.abs(A[sample]) @ np.abs(B))
    assert np.all(np.abs(got - A[sample] @ B) <= bound)


# exponents of the tiny and the huge operand: the tiny one's third piece is
# dropped in part, the second one too, and almost all of it
@pytest.mark.parametrize("tiny,huge", [(-118, 62), (-127, 98), (-134, 108)])
@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(129, 200, 70), (4096, 256, 130), (64, 576, 5000)] + TILES, ids=IDS)
def test_tiny_times_huge(hip, layout, shape, tiny, huge):
    """Bits that the split of a tiny operand drops matter as much as the other
    operand makes them, with results of any size."""
    rows, cols, inner = shape
    rng = np.random.default_rng(11 * rows + layout - tiny)
    small = lambda s: np.ldexp(rng.standard_normal(s), tiny).astype(np.float32)
    large = lambda s: np.ldexp(rng.standard_normal(s), huge).astype(np.float32)
    sample = np.unique(np.linspace(0, rows - 1, 97).astype(int))
    for ma, mb in ((small, large), (large, small)):
        a, b = operands(layout, rows, cols, inner, ma, mb)
        A, B = logical(layout, a, b)
        got = gemm(hip, layout, a, b, rows, cols, inner)[sample]
        # (f32 instructions round every product and sum)
        bound = (inner + 8) * 2.0 ** -24 * (np.abs(A[sample]) @ np.abs(B))
        assert np.all(np.abs(got - A[sample] @ B) <= bound)


def test_tiny_times_huge_in_a_group(hip):
    """The products of a Linear's backward, which share one launch: a single
    tiny value of a row that is otherwise zero, and of a column."""
    rng = np.random.default_rng(3)
    batch, in_f, out_f = 4096, 128, 192
    x = rng.standard_normal((batch, in_f)).astype(np.float32)
    w = np.ldexp(rng.standard_normal((in_f, out_f)), 90).astype(np.float32)
    g = np.zeros((batch, out_f), np.float32)
    g[5, 7], g[77, 100], g[4000] = 1.2345678e-36, 2.0 ** -129 * 1.37, np.float32(1.2345678e-38)
    x[5] *= np.float32(2.0 ** 80)
    dx, dw = hip.DeviceBuffer(batch * in_f), hip.DeviceBuffer(in_f * out_f)
    hip.call("nrs_linear_backward", dx, dw, None, hip.DeviceBuffer.from_host(g),
             hip.DeviceBuffer.from_host(x), hip.DeviceBuffer.from_host(w), batch, in_f, out_f, 0.0, 0.0, 0.0)
    X, W, G = (v.astype(np.float64) for v in (x, w, g))
    for got, want, size, k in ((dx.to_host((batch, in_f)), G @ W.T, np.abs(G) @ np.abs(W.T), out_f),
                               (dw.to_host((in_f, out_f)), X.T @ G, np.abs(X.T) @ np.abs(G), batch)):
        # (2^-149: results under f32's smallest normal value)
        assert np.all(np.abs(got - want) <= (k + 8) * 2.0 ** -24 * size + k * 2.0 ** -149)


@pytest.mark.parametrize("layout", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(129, 200, 70), (4096, 256, 130), (64, 576, 5000)] + TILES, ids=IDS)
def test_bits_do_not_depend_on_other_rows_and_columns(hip, layout, shape):
    """Rows of A and columns of B with values that the split cannot hold change
    no bit of the other rows' and columns' results."""
    rows, cols, inner = shape
    rng = np.random.default_rng(rows + layout)
    make = lambda s: rng.standard_normal(s).astype(np.float32)
    a, b = operands(layout, rows, cols, inner, make, make)
    before = gemm(hip, layout, a, b, rows, cols, inner)
    A, B = (a.T if layout == TN else a), (b.T if layout == NT else b)  # views
    odd = [3, 40, rows - 2]
    A[3, 5], A[40] = np.nan, np.inf
    A[rows - 2] *= np.float32(2.0 ** -119)
    B[1, cols - 3], B[:, 20] = np.float32(3.4e38), np.float32(2.0 ** -127 * 1.3)
    after = gemm(hip, layout, a, b, rows, cols, inner)
    same = np.ones((rows, cols), bool)
    same[odd] = False
    same[:, [20, cols - 3]] = False
    assert np.array_equal(before[same], after[same])


def test_bmm_large_items(hip):
    """Batched items past the small-item kernel, each at its own offset."""
    rng = np.random.default_rng(1)
    batch, m, n, k = 5, 150, 131, 77
    a, b = int_matrix(rng, (batch, m, k)), int_matrix(rng, (batch, k, n))
    c = hip.DeviceBuffer(batch * m * n)
    hip.bmm(NN, c, hip.DeviceBuffer.from_host(a), hip.DeviceBuffer.from_host(b), batch, m, n, k)
    assert np.array_equal(c.to_host((batch, m, n)), a @ b)


@pytest.mark.parametrize("batch,in_f", [(4096, 256), (500, 128), (300, 100)])
def test_row_of_sums(hip, batch, in_f):
    """A weight gradient alone, with its bias gradient as a row of sums (a tile
    row of its own where in_f is a multiple of 64)."""
    rng = np.random.default_rng(batch)
    out_f = 192
    x, g = int_matrix(rng, (batch, in_f), -2, 2), int_matrix(rng, (batch, out_f), -2, 2)
    dw, db = hip.DeviceBuffer(in_f * out_f), hip.DeviceBuffer(out_f)
    hip.call("nrs_linear_backward", None, dw, db, hip.DeviceBuffer.from_host(g),
             hip.DeviceBuffer.from_host(x), None, batch, in_f, out_f, 0.0, 0.0, 0.0)
    assert np.array_equal(dw.to_host((in_f, out_f)), x.T @ g)
    assert np.array_equal(db.to_host(), g.sum(0))
