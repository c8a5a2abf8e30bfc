"""Convolutions on the split tiles (conv_split.hip), against f64.

Shapes take every tile and every staging form where it can go wrong: channels
that are and are not whole k steps, ragged channel and pixel tiles, rows of
whole quads (128-bit loads, moved one pixel at the image's edges) and ragged
rows, strides, padding 0 and past 1, 1x1 and 5x5 kernels, few-channel weight
gradients, pointers off 16 bytes.

plan.CONV_TILES has layers that reach the wide tiles of the forward and the
input gradient (checked on the CPU).

Bars: bit-exact where every product and partial sum is an integer below 2^24
(one operand of up to 16 bits, so that every piece carries bits); against f64,
|y - y64| <= (6 K / 16 + 72) * 2^-24 * (|x| * |w|) element by element: the split
tiles round their large accumulator K / 8 times and the other one, 2^-7 of it,
5 K / 8 times, and drop and leave out at most 9 units (test_gpu_gemm_split.py),
and a weight gradient's partial sums (at most 64 long a chain) and its beta
round too. (The f32 kernels that take some of the layers round K times, but
hold this bar.)
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import plan
from kat import int_matrix

pytestmark = pytest.mark.gpu

SHAPES = [  # n, c_in, c_out, h, w, kh, kw, stride, pad
    (2, 64, 64, 24, 24, 3, 3, 1, 1),     # whole k steps and tiles, 128-bit window loads
    (3, 64, 72, 17, 19, 3, 3, 1, 1),     # ragged rows, ragged channel tile
    (9, 36, 65, 21, 20, 3, 3, 1, 1),     # channels across k steps, pixels across images
    (40, 128, 128, 21, 21, 3, 3, 1, 1),  # whole k steps over pixels across images
    (2, 64, 48, 23, 20, 3, 3, 1, 0),     # no padding
    (2, 64, 40, 18, 18, 3, 3, 1, 2),     # padding past 1
    (2, 64, 64, 20, 20, 5, 5, 1, 2),
    (2, 40, 72, 30, 28, 1, 1, 1, 0),
    (2, 64, 36, 31, 33, 3, 3, 2, 1),
    (2, 32, 64, 32, 32, 3, 3, 2, 1),     # strided, rows of whole quads
    (2, 64, 64, 12, 40, 2, 4, 1, 1),     # kernel and image not square
    (4, 3, 32, 32, 32, 3, 3, 1, 1),      # weight gradient of 27 columns
    (4, 3, 96, 30, 29, 3, 3, 2, 1),
    (2, 1, 96, 28, 28, 3, 3, 1, 1),
    (2, 16, 20, 40, 40, 3, 3, 1, 1),     # 145 columns, 20 rows
    (2, 16, 32, 41, 39, 3, 3, 1, 1),     # 32-row tiles full, ragged rows of pixels
    (4, 128, 1, 24, 24, 1, 1, 1, 0),     # one channel, 129 columns
    (2, 8, 33, 40, 40, 4, 4, 1, 1),      # a row and a column past them (33, 129)
    (4, 8, 32, 48, 48, 4, 4, 2, 1),      # 129 columns, strided rows of whole quads
    (4, 24, 24, 30, 30, 5, 5, 2, 2),     # 601 columns, strided ragged rows
    # a few k steps in all (not a "same" layer: Winograd's sums, which such small
    # ones take, cancel, and its error has no bound element by element)
    (1, 16, 32, 5, 6, 3, 3, 1, 0),
    (1, 9, 70, 1, 4, 3, 3, 1, 1),        # one output row of one quad
    (3, 256, 160, 7, 7, 3, 3, 1, 1),     # the sum of 6 slices, 8 waves a group
    (2, 48, 70, 8, 12, 3, 3, 2, 1),      # of 2 slices, two groups a workgroup
    (3, 48, 70, 8, 12, 3, 3, 2, 1),      # of 3, a wave of four with none
    # layers that the rules leave to the kernels before the split tiles: a weight
    # gradient of few columns, of many over few pixels, and the backward pair
    (30, 4, 8, 21, 23, 1, 1, 1, 0),
    (2, 64, 128, 6, 5, 5, 5, 1, 2),
    (1, 16, 128, 20, 20, 3, 3, 1, 1),
]
WIDE = [shape for shape, _, _ in plan.CONV_TILES]
IDS = lambda s: "x".join(map(str, s))


def device(hip, x, offset):
    buf = hip.DeviceBuffer.from_host(np.concatenate([np.zeros(offset, np.float32), x.ravel()]))
    return buf, buf.ptr + 4 * offset


def reference(shape, x, w, b, g):
    n, ci, co, h, wd, kh, kw, s, p = shape
    tx, tw, tb = (torch.from_numpy(v.astype(np.float64)).requires_grad_() for v in (x, w, b))
    y = F.conv2d(tx, tw, tb, stride=s, padding=p)
    y.backward(torch.from_numpy(g.astype(np.float64)))
    return [v.detach().numpy() for v in (y, tx.grad, tw.grad, tb.grad)]


def run(hip, shape, x, w, b, g, old, beta_in, beta_par, offset=0, dinput=True):
    n, ci, co, h, wd, kh, kw, s, p = shape
    dims = (n, ci, h, wd, co, kh, kw, s, p)
    keep = [device(hip, v, offset) for v in (x, w, b, g)]
    px, pw, pb, pg = (k[1] for k in keep)
    y = hip.DeviceBuffer.from_host(np.full(g.size, np.nan, np.float32))
    hip.call("nrs_conv2d_forward", y.ptr, px, pw, pb, *dims)
    dx, dw, db = (hip.DeviceBuffer.from_host(v) for v in old)
    hip.call("nrs_conv2d_backward_ex", dx.ptr if dinput else None, dw.ptr, db.ptr, pg, px, pw, *dims,
             beta_in, beta_par)
    return y.to_host(g.shape), dx.to_host(x.shape), dw.to_host(w.shape), db.to_host(b.shape)


def sizes(shape):
    n, ci, co, h, w, kh, kw, s, p = shape
    oh, ow = (h + 2 * p - kh) // s + 1, (w + 2 * p - kw) // s + 1
    return (n, ci, h, w), (co, ci, kh, kw), (co,), (n, co, oh, ow)


@pytest.mark.parametrize("shape", SHAPES + WIDE, ids=IDS)
def test_exact_integers_all_pieces(hip, shape):
    sx, sw, sb, sg = sizes(shape)
    rng = np.random.default_rng(sum(shape))
    longest = max(sw[1] * sw[2] * sw[3], sw[0] * sw[2] * sw[3], sg[0] * sg[2] * sg[3])
    bits = min(16, 23 - int(np.ceil(np.log2(longest))))
    wide = lambda s: int_matrix(rng, s, -2 ** bits + 1, 2 ** bits - 1)
    sign = lambda s: int_matrix(rng, s, -1, 1)
    # (the input gradient is g * w, the weight gradient g * x)
    for offset, (mx, mw, mg) in enumerate([(wide, sign, sign), (sign, wide, sign), (sign, sign, wide)]):
        x, w, b, g = mx(sx), mw(sw), sign(sb), mg(sg)
        old = [sign(sx), sign(sw), sign(sb)]
        got = run(hip, shape, x, w, b, g, old, 1.0, 1.0, offset)
        want = reference(shape, x, w, b, g)
        for k, name in enumerate(("output", "input gradient", "weight gradient", "bias gradient")):
            assert np.array_equal(got[k].astype(np.float64), want[k] + (old[k - 1] if k else 0)), name


@pytest.mark.parametrize("shape", SHAPES + WIDE, ids=IDS)
def test_f64_error(hip, shape):
    sx, sw, sb, sg = sizes(shape)
    rng = np.random.default_rng(3 + sum(shape))
    # magnitudes over nine decades, one value in three zero
    make = lambda s: (rng.standard_normal(s) * 10.0 ** rng.integers(-6, 4, s) *
                      (rng.random(s) > 0.33)).astype(np.float32)
    x, w, b, g = make(sx), make(sw), make(sb), make(sg)
    nan = [np.full(s, np.nan, np.float32) for s in (sx, sw, sb)]
    got = run(hip, shape, x, w, b, g, nan, 0.0, 0.0, dinput=False)
    grads = run(hip, shape, x, w, b, g, nan, 0.0, 0.0)
    assert np.isnan(got[1]).all()  # no input gradient asked for
    want, size = reference(shape, x, w, b, g), reference(shape, *map(np.abs, (x, w, b, g)))
    ks = (sw[1] * sw[2] * sw[3], sw[0] * sw[2] * sw[3], sg[0] * sg[2] * sg[3], sg[0] * sg[2] * sg[3])
    for k, name in enumerate(("output", "input gradient", "weight gradient", "bias gradient")):
        bound = (6 * ks[k] / 16 + 72) * 2.0 ** -24 * size[k] + 1e-35
        for y in ((grads[k],) if k == 1 else (got[k], grads[k])):
            assert np.all(np.abs(y - want[k]) <= bound), name


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[1], SHAPES[3], SHAPES[9], SHAPES[11]] + WIDE, ids=IDS)
def test_infinities_and_nan_stay_where_they_belong(hip, shape):
    sx, sw, sb, sg = sizes(shape)
    rng = np.random.default_rng(5 + sum(shape))
    small = lambda s: int_matrix(rng, s, 1, 4)
    x, w, b, g = small(sx), small(sw), small(sb), small(sg)
    x[0, 1, 2, 3], x[-1, 0, -1, -1] = np.inf, np.float32(3.4028235e38)
    # (the values that are not finite meet no padding: a lowering's padding zeros
    # times them are NaN, where torch has no such term)
    mid = shape[5] // 2, shape[6] // 2
    w[(5, 0) + mid] = np.nan
    w[(3, 1) + mid] = 2.0 ** -100
    g[0, 2, 1, 1], g[-1, 1, -2, -2] = -np.inf, np.nan
    old = [np.zeros(s, np.float32) for s in (sx, sw, sb)]
    got = run(hip, shape, x, w, b, g, old, 0.0, 0.0)
    want = reference(shape, x, w, b, g)
    for k in range(4):
        with np.errstate(over="ignore"):
            f = want[k].astype(np.float32)
        bad = ~np.isfinite(f)
        assert not np.isfinite(got[k][bad]).any()
        ok = ~bad
        assert np.all(np.abs(got[k][ok] - f[ok]) <= 1e-4 * np.abs(f[ok]) + 1e-30)


@pytest.mark.parametrize("tiny", range(3))
@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[1], SHAPES[3], SHAPES[8], SHAPES[11], SHAPES[15]] + WIDE,
                         ids=IDS)
def test_tiny_times_huge(hip, shape, tiny):
    """One of image, weights and gradient below the split's exact range, the
    others large: the bits it drops would show in results of any size."""
    sx, sw, sb, sg = sizes(shape)
    rng = np.random.default_rng(7 + sum(shape) + tiny)
    make = lambda s, e: np.ldexp(rng.random(s) + 0.5, e).astype(np.float32)
    x, w, g = (make(s, -118 if i == tiny else 54) for i, s in enumerate((sx, sw, sg)))
    b = np.zeros(sb, np.float32)
    nan = [np.full(s, np.nan, np.float32) for s in (sx, sw, sb)]
    got = run(hip, shape, x, w, b, g, nan, 0.0, 0.0)
    want, size = reference(shape, x, w, b, g), reference(shape, *map(np.abs, (x, w, b, g)))
    ks = (sw[1] * sw[2] * sw[3], sw[0] * sw[2] * sw[3], sg[0] * sg[2] * sg[3], sg[0] * sg[2] * sg[3])
    for k, name in enumerate(("output", "input gradient", "weight gradient", "bias gradient")):
        # (f32 instructions round every product and sum)
        bound = (ks[k] + 72) * 2.0 ** -24 * size[k]
        assert np.all(np.abs(got[k] - want[k]) <= bound), name


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[1], SHAPES[3], SHAPES[8]] + WIDE[:4], ids=IDS)
def test_bits_do_not_depend_on_the_other_images(hip, shape):
    """An image of values that the split cannot hold changes no bit of the
    other images' outputs and input gradients."""
    sx, sw, sb, sg = sizes(shape)
    rng = np.random.default_rng(13 + sum(shape))
    make = lambda s: rng.standard_normal(s).astype(np.float32)
    x, w, b, g = make(sx), make(sw), make(sb), make(sg)
    nan = [np.full(s, np.nan, np.float32) for s in (sx, sw, sb)]
    y0, dx0, _, _ = run(hip, shape, x, w, b, g, nan, 0.0, 0.0)
    x[-1, :, 2] *= np.float32(2.0 ** -119)
    x[-1, 0, 0, 0], g[-1, 1, 0, 0] = np.inf, np.nan
    g[-1, :, -1] *= np.float32(2.0 ** -125)
    y1, dx1, _, _ = run(hip, shape, x, w, b, g, nan, 0.0, 0.0)
    assert np.array_equal(y0[:-1], y1[:-1]) and np.array_equal(dx0[:-1], dx1[:-1])
