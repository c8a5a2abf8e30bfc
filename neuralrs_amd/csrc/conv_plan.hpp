// What the convolution kernels are asked for, and which of them takes a layer.
// Host only and free of HIP, so that a CPU test can ask.
//
// out[n, m, oy, ox] = sum_{c,i,j} x[n, c, oy*s - pad_h + i, ox*s - pad_w + j] * Wt(m, c, i, j)
//                     (+ bias[m]) + beta * out
// with Wt(m, c, i, j) = w[m][c][i][j] (forward), or, with `flip`, the
// flipped, channel-transposed w[c][m][kh-1-i][kw-1-j] (the stride-1 input
// gradient of a convolution with weights w, read as a forward convolution of
// the output gradient).
#pragma once

#include <cstdint>

#include "gemm_plan.hpp"

namespace nrs {

struct SlabConv {
    const float* x = nullptr;     // NCHW [N][C][H][W]
    const float* w = nullptr;     // [M][C][kh][kw], or [C][M][kh][kw] with flip
    const float* bias = nullptr;  // [M] or null
    float* out = nullptr;         // NCHW [N][M][OH][OW]
    int64_t N = 0;
    int C = 0, H = 0, W = 0, M = 0, kh = 0, kw = 0, stride = 1, pad_h = 0, pad_w = 0;
    int OH = 0, OW = 0;
    bool flip = false;
    float beta = 0.0f;
};

// Weight gradient dw[m][c][i][j] += sum g[n,m,oy,ox] * x[n,c,oy*s-pad+i,ox*s-pad+j]
// and, when db is given, bias gradient db[m] += sum g[n,m,oy,ox].
struct SlabWgrad {
    const float* x = nullptr;  // NCHW [N][C][H][W]
    const float* g = nullptr;  // NCHW [N][M][OH][OW]
    float* dw = nullptr;       // [M][C][kh][kw]
    float* db = nullptr;       // [M] or null
    int64_t N = 0;
    int C = 0, H = 0, W = 0, M = 0, kh = 0, kw = 0, stride = 1, pad = 0, OH = 0, OW = 0;
    float beta = 1.0f;  // dw = gradient + beta * dw (likewise db); 0 reads nothing
};
// Whether the split tiles (conv_split.hip) can take a convolution: whole quads of
// channels, the taps of the padded last k step within a 32-bit mask, an image
// within 32-bit offsets, and more than 32 output channels.
inline bool split_conv_takes(const SlabConv& s) {
    const int64_t taps = (int64_t)s.kh * s.kw, pixels = s.N * s.OH * s.OW;
    const int64_t in_bytes = s.N * s.C * s.H * s.W * 4 + ((int64_t)s.pad_h * s.W + s.pad_w) * 4;
    return s.C > 0 && s.C % 4 == 0 && cdiv(taps * s.C, 64) * 64 / s.C <= 31 && s.M > 32 &&
           pixels >= 64 && pixels <= INT32_MAX && in_bytes <= 0x7fffffffll &&
           (int64_t)s.M * s.C * taps <= (1 << 28) && s.pad_h >= 0 && s.pad_w >= 0;
}

// The tile they take it on (there is no 256x256 one).
inline int split_conv_tile(const SlabConv& s, int cus) {
    const int tile = cheapest_split_tile(s.M, s.N * s.OH * s.OW, (int64_t)s.C * s.kh * s.kw, 1, true, cus);
    return tile == S256x256 ? (int)S128x128 : tile;
}

// Whether the split tiles take a convolution ahead of the kernels that hold
// their operands in LDS (split_conv may still refuse it). It is an estimate
// against each, us on both sides, from sweeps over 8 .. 256 channels, 7x7 ..
// 64x64 images and batches of 1 .. 256:
// - small "same" 3x3 images, whose kernels give an image and a block of
//   outputs to a workgroup, so they take whole rounds of the CUs whatever the
//   image holds: N 64 128->128 14^2 36 against 45 (kept), 8^2 34 / 25, N 256
//   256->256 8^2 492 / 112, N 8 64->64 14^2 20 / 16.5;
// - the slab kernel is ahead by its one launch less where the reduction and
//   the output are short: 16->40 32^2 13.4 / 17.0, 24->64 32^2 18.6 / 19.9,
//   16->128 1x1 64^2 15.4 / 19.3, but 64->64 32^2 79 / 27, 48->64 64^2 138 / 68.
//   Under 16 channels of 9 taps it stays ahead over any number of pixels (64
//   outputs, N 256: 16 channels 20^2 32.0 / 36.9, 8 channels 16^2 15.0 / 18.7),
//   under 24 up to the 65536 of N 256 16^2 (21.4 / 26.5), and 64->64 1x1 20^2
//   (N 256 23 / 25). Over few pixels a long reduction leaves the split tiles a
//   chain of k steps on part of the chip: 32->64 5x5 N 64 10^2 17.5 / 22.7,
//   64->64 stride 2 N 64 10^2 15.2 / 17.5.
// (Two workgroups of the odd images' kernel fit a CU: 16->64 5^2 N 128 takes
// one round, 6.6 against 12.3.)
inline bool split_conv_better(const SlabConv& s, int cus) {
    const int64_t taps = (int64_t)s.kh * s.kw, K = s.C * taps, px = s.N * s.OH * s.OW;
    if (s.M <= 64 && (taps == 1 ? K <= 64
                                : K <= 144 ? s.stride == 1 || px > 32768
                                : K <= 216 && s.stride == 1 ? px <= 65536
                                : taps > 9 ? px <= 8192 : s.stride > 1 && K <= 576 && px <= 2048))
        return false;
    if (taps == 9 && s.kh == 3 && s.stride == 1 && s.OH == s.H && s.OW == s.W && s.H <= 16 && s.W <= 16 &&
        s.C % 16 == 0 && s.M % 32 == 0) {
        const double small = s.W % 2 == 0 ? (double)((s.N * (s.M / 32) + cus - 1) / cus) * (4.5 + 0.225 * s.C)
                                          : (double)((s.N * (s.M / 16) + 2 * cus - 1) / (2 * cus)) * (3.5 + 0.165 * s.C);
        double split;
        cheapest_split_tile(s.M, px, K, 1, true, cus, &split);
        return split + 7.0 < small;  // (packing the weights, staging the windows)
    }
    return K > 32 && !(taps > 1 && K <= 448 && (((s.M <= 48 || (s.stride == 1 && s.M <= 64)) && px <= 32768) ||
                                    (s.stride == 1 && px <= 16384)));
}

// Whether the chunk-pipelined backward (pipe_backward, where its geometry
// holds) is ahead of the split tiles: narrow layers, while a round of its
// workgroups does not outlast the images' own work. Both gradients, pipelined
// against split (us): N 64 32->64 14^2 28 / 44, 64->64 14^2 31 / 45, N 256
// 64->64 14^2 92 / 89, 8^2 79 / 42, N 64 128->128 14^2 114 / 93, 8^2 96 / 51.
// The weight gradient alone is ahead with enough images: N 64 64->64 14^2
// 28 / 29, N 8 25 / 15, N 256 32->64 8^2 19 / 22, 10^2 22 / 31, 64->64 10^2
// 36 / 40, 8^2 32 / 27.
inline bool pipe_backward_better(const SlabWgrad& w, bool dinput) {
    if (w.C > 64 || w.M > 64) return false;
    if (dinput) return w.N <= 128 || w.H * w.W > 100;
    return w.N >= 64 && (w.N <= 128 || w.H * w.W >= 100 || w.C <= 32);
}

// Whether the direct weight gradient of few columns (small_wgrad, a workgroup an
// image and 4, 2 or 1 channels) is ahead of the split tiles, where 64 channels
// and 64 columns cost the same however few there are. Both are estimated in us,
// fitted to 1777 layers of 1 .. 32 columns, 4 .. 128 channels, images 7x7 ..
// 64x64 and batches of 1 .. 256: the choice is 0.8% from the better one in the
// mean, and the split tiles alone 4.7%, up to three times: 4->8 1x1 N 208 37^2
// 14.5 / 44, 1->16 3x3 N 218 63^2 46 / 108, 1->32 N 161 63^2 1x1 53 / 85, but
// 3->32 3x3 N 32 64^2 121 / 21. The direct kernel has to be ahead by more than the
// fits are usually wrong: of 372 other layers where it was by any margin, 27 were
// 5 to 40% slower (4->128 1x1 N 205 37^2 120 / 85), by 7% 6.
inline bool small_wgrad_better(const SlabWgrad& w) {
    const int64_t taps = (int64_t)w.C * w.kh * w.kw, P = (int64_t)w.OH * w.OW;
    if (w.N * w.M * (taps + 1) > INT32_MAX) return false;  // (small_wgrad's partials)
    const int cls = taps <= 9 ? 0 : taps <= 16 ? 1 : 2, channels = 4 >> cls;
    const double base[3] = {7.2, 8.9, 10.8}, round[3] = {1.28, 2.6, 5.07}, image[3] = {1.9, 6.1, 7.6};
    const double groups = (double)(w.N * ((w.M + channels - 1) / channels)) / 256, kpx = (double)P / 1000;
    const double small = base[cls] + round[cls] * groups * (1 + kpx) + image[cls] * kpx;
    const int64_t quads = w.N * w.OH * ((w.OW + 3) / 4);
    const double step = w.OW % 4 ? 1.06 : w.stride == 1 && w.pad <= 1 && w.W >= 4 ? 0.7 : 0.88;
    const double split = 9.2 + step * (double)((w.M + 63) / 64) * (double)quads / (8 * 256);
    return small < 0.93 * split;
}

// Whether the im2col lowering (three launches) of a weight gradient past the
// slab kernel's 18 taps is ahead of the split tiles: a large output over a few
// hundred pixels, where tiles, partial sums and their launch are all there is.
// 5x5, im2col against split (us): 256->256 N 2 5^2 14.5 / 23, 128->256 N 1 21^2
// stride 2 14.6 / 23, 128->128 N 1 24^2 22 / 19, 256->256 N 3 19^2 60 / 36.
inline bool im2col_wgrad_better(const SlabWgrad& w) {
    const int64_t taps = (int64_t)w.kh * w.kw;
    return taps > 18 && w.N * w.OH * w.OW <= 400 && w.M * (w.C * taps + 1) >= 1 << 17;
}

// Whether the slab weight gradient on its own is: many small images, above all
// of rows that are no whole quads, whose pixels the split tiles gather one by
// one. Slab against split (us): N 256 16->32 7^2 15 / 18; 10^2 N 128 32->32
// 18 / 21, N 256 16->64 20 / 26, N 64 32->32 17 / 15; 9^2 N 100 32->32 17 / 19;
// 14^2 N 128 24->64 25 / 28,
// N 256 16->64 26 / 32, 64->32 59 / 50; of quads, 12^2 N 256 32->32 28 / 25.
inline bool slab_wgrad_better(const SlabWgrad& w) {
    const int64_t pixels = (int64_t)w.H * w.W;
    if (w.kh * w.kw > 9 || w.stride != 1 || pixels > 196) return false;
    if (w.N > 128 && w.C * w.M <= 512) return true;
    return w.OW % 4 != 0 && pixels >= 81 && w.C >= 16 && w.C <= 32 && w.N >= 96;
}

// Whether the slab pair is: narrow layers over small images, where one launch
// of both gradients fills the chip that neither does alone. Up to 14x14 an
// image is one band, and the pair's time is mostly its launches' until images
// times products, the input channels counted twice (they are the output rows of
// one half and the columns of the other), outgrow the chip. Pair against split
// (us): 14^2 N 128 16->64 30 / 41, 32->32 30 / 39, 64->32 51 / 47; 10^2 N 64
// 8->64 19 / 28, N 256 16->64 28 / 41, 64->16 49 / 46; 8^2 N 64 32->32 17 / 23,
// N 256 64->20 48 / 40. Larger images come in bands: 16^2 N 64 32->64 33 / 41,
// 8->64 30 / 29, N 128 43 / 33. Up to 32 input channels the split tiles do not
// take the input gradient, and on its own over many gradient channels it is one
// long chain a workgroup: 32->96 N 24 15^2 37 / 66, N 8 40^2 47 / 57. With up to
// 16 it stays ahead, of more than 96 gradient channels, until the gradient
// outgrows the pair's launch: 8->256 N 4 45^2 61 / 83, 16->128 N 1 20^2 37 / 50, but
// 8->256 N 16 32^2 98 / 80. Up to 96 are one and a half of the split weight
// gradient's 64-row tiles and little work for the input gradient's chain: there
// the pair gains over a few large images, 16->96 N 2 54^2 41 / 55, and loses over
// less or over small ones, 8->96 N 2 25^2 47 / 33, N 31 31^2 63 / 46.
inline bool slab_pair_better(const SlabWgrad& w) {
    const int64_t pixels = (int64_t)w.H * w.W, size = (int64_t)w.C * w.C * w.M * w.N;
    const int taps = w.kh * w.kw;
    if (taps > 9 || w.stride != 1) return false;
    if (taps > 1 && w.M > 64 && w.C > 16 && w.C <= 32 && w.N * pixels <= 16384) return true;
    if (taps > 1 && w.M > 64 && w.C <= 16 && w.N * pixels * w.M <= 5 << 19 &&
        (w.M > 96 || (w.N * pixels > 6144 && pixels >= 1296)))
        return true;
    if (w.H > 16 || w.W > 16) return false;
    if (pixels <= (w.OW % 4 ? 225 : 196) && size <= (taps == 1 && pixels <= 100 ? 20 : 15) << 20) return true;
    if (w.C * w.M <= 512) return pixels <= 64 || (w.N > 128 && pixels <= 196);
    return w.C * w.M <= 2048 && pixels > 196 && size <= (1 << 22);
}

}  // namespace nrs
