// Convolutions as implicit GEMMs on the split tiles (gemm_split.hpp): f32
// operands gathered from NCHW in place, split into bf16 pieces while staged.
// Replaces im2col + matmul + col2out (src/cuda/nn/conv.rs:266-277), the
// stride-1 input gradient (:304-312) and the weight and bias gradient
// (:314-322) for layers whose images do not fit the small-image kernels.
//
// Forward, and the stride-1 input gradient as the flipped convolution of the
// output gradient: rows are output channels, columns output pixels, and the
// reduction runs tap by tap, channels inside (k = tap * C + c). A staging unit
// is 4 + 4 consecutive k of one pixel, so with C % 4 == 0 each half lies in
// one tap: its padding test is one bit of a per-pixel mask of taps, its eight
// addresses are the pixel's offset plus scalars, and gathering costs about as
// much as a dense operand (the lanes run along the pixels). The weights are
// read in their own layout the same way.
//
// Weight gradient: rows are output channels, columns (c, tap) pairs and one
// column of ones (the bias gradient), and the reduction runs over pixels in
// quads of one output row (rows padded to whole quads, the padding zero in
// the gradient operand). Four lanes stage the units of a row, each finding its
// two quads' image and row once a k-tile. K slices write partial tiles and one
// launch adds them in slice order.
//
// What bounds them: gathering. A forward k step of a 64 x 128 tile takes about
// 1.1 us, 0.9 with dense operands; the weight gradient's window loads are 128
// bits only where rows are whole quads. Against the f32 slab kernels (us, 3x3
// of stride 1 unless said):
//   forward      64->128 32 x 32^2 117 -> 38    128->128 64 x 28^2 225 -> 108
//                64->64 5x5 32 x 32^2 135 -> 58   64->128 stride 2 32 x 56^2 66 -> 37
//   wgrad + bias 16->32 32 x 64^2 75 -> 34   64->128 32 x 32^2 122 -> 44
//                128->128 64 x 28^2 310 -> 104   3->32 32 x 64^2 121 -> 21
//                1x1 64->128 32 x 32^2 101 -> 20
#include <algorithm>
#include <cmath>

#include "conv_slab.hpp"
#include "gemm_call.hpp"
#include "gemm_split.hpp"

namespace nrs {
namespace {

struct ConvSplitArgs {
    GemmArgs g;  // A weights (output gradient), B image; M, N, K, epilogue
    int C, H, W, taps, kw, stride, pad_h, pad_w, OH, OW;
    int quads;         // weight gradient: pixel quads in all
    FastDiv div_c, div_kw, div_p, div_ow;  // C, kw, OH * OW, OW
    FastDiv div_rowq, div_oh, div_taps;    // quads of a row, OH, taps
};

// ------------------------------------------------ forward / input gradient

// The weights as the dense operand [m][k = tap * C + c] from [m][c][tap], or,
// flipped, from [c][m][taps - 1 - tap]: read in place, the lanes of a load
// would be a row apart (32 -> 64 channels over 32 x 32: 26 us against 17).
__global__ __launch_bounds__(256) void conv_split_weights_kernel(float* dst, const float* w, int M,
                                                                 int C, int taps, int flip,
                                                                 FastDiv div_c, FastDiv div_taps) {
    const int total = M * C * taps;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < total; e += gridDim.x * 256) {
        uint32_t mt, c, m, t;
        fast_divmod((uint32_t)e, div_c, mt, c);
        fast_divmod(mt, div_taps, m, t);
        dst[e] = flip ? w[((int)c * M + (int)m) * taps + taps - 1 - (int)t]
                      : w[((int)m * C + (int)c) * taps + (int)t];
    }
}

// The im2col matrix of the image: pixels along the lanes.
// ONE_TAP: C is a multiple of BK, so a k-tile lies in one tap.
template <int BN, int BK, int NT, int U, bool ONE_TAP>
struct ConvPixels {
    static constexpr bool kKC = false, kOnes = false, kMasked = true, kFix = false;
    static constexpr uint32_t ones = 0;
    const ConvSplitArgs* a;
    const float* base;  // the image, one padding corner before its start
    int64_t n0;
    int off;        // bytes of the thread's pixel (its window's corner)
    uint32_t mask;  // bit tap: the pixel's window has that tap inside the image
    int tile_off, tile_s;  // ONE_TAP: the k-tile's vector offset and scalar offset of its channel 0

    __device__ __forceinline__ void corner(int64_t n, int& img, int& iy0, int& ix0) const {
        uint32_t im, p, oy, ox;
        fast_divmod((uint32_t)min(n, a->g.N - 1), a->div_p, im, p);
        fast_divmod(p, a->div_ow, oy, ox);
        img = (int)im;
        iy0 = (int)oy * a->stride - a->pad_h;
        ix0 = (int)ox * a->stride - a->pad_w;
    }
    __device__ __forceinline__ void init(const ConvSplitArgs& args, int64_t n0_, int tid) {
        static_assert(NT % BN == 0 && BN % 64 == 0, "one pixel a thread, one unit index a wave");
        a = &args;
        n0 = n0_;
        const int corner0 = a->pad_h * a->W + a->pad_w;
        base = a->g.B - corner0;
        int img, iy0, ix0;
        corner(n0 + tid % BN, img, iy0, ix0);
        off = (img * a->C * a->H * a->W + iy0 * a->W + ix0 + corner0) * 4;
        mask = 0;
        for (int t = 0, i = 0, j = 0; t < a->taps; ++t) {
            const bool in = ((unsigned)(iy0 + i) < (unsigned)a->H) & ((unsigned)(ix0 + j) < (unsigned)a->W);
            mask |= (uint32_t)in << t;
            if (++j == a->kw) {
                j = 0;
                ++i;
            }
        }
    }
    __device__ __forceinline__ int tap_s(uint32_t tap, uint32_t c) const {
        uint32_t ti, tj;
        fast_divmod(tap, a->div_kw, ti, tj);
        return __builtin_amdgcn_readfirstlane(((int)c * a->H * a->W + (int)ti * a->W + (int)tj) * 4);
    }
    __device__ __forceinline__ int tap_off(uint32_t tap) const {  // (tap < 32)
        return ((mask >> tap) & 1u) ? off : kOutOfRange;
    }
    __device__ __forceinline__ void begin(int64_t k0, int) {
        if constexpr (ONE_TAP) {
            uint32_t tap, c;
            fast_divmod((uint32_t)__builtin_amdgcn_readfirstlane((int)k0), a->div_c, tap, c);
            tile_s = tap_s(tap, c);
            tile_off = tap_off(tap);
        }
    }
    __device__ __forceinline__ void fix(f32x4 (&)[2], int) const {}
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&r)[2], int i, int64_t k0, int64_t, int tid) const {
        const int q = __builtin_amdgcn_readfirstlane((tid + i * NT) / BN);
        const auto rsrc = buffer_rsrc(base, 0x80000000ll);
        const int plane4 = a->H * a->W * 4;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int kk = half * (BK / 2) + 4 * q;
            int s0, voff;
            if constexpr (ONE_TAP) {
                s0 = tile_s + kk * plane4;
                voff = tile_off;
            } else {
                uint32_t tap, c;
                fast_divmod((uint32_t)__builtin_amdgcn_readfirstlane((int)k0 + kk), a->div_c, tap, c);
                s0 = tap_s(tap, c);
                voff = tap_off(tap);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                r[half][e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff, s0 + e * plane4, 0));
        }
    }
    struct Spot {
        int off, iy0, ix0;  // bytes of the pixel's window corner, and where it lies
    };
    __device__ __forceinline__ Spot spot(int col) const {
        int img, iy0, ix0;
        corner(n0 + col, img, iy0, ix0);
        return Spot{(img * a->C * a->H * a->W + (iy0 + a->pad_h) * a->W + ix0 + a->pad_w) * 4, iy0, ix0};
    }
    template <bool PART>  // (K is a multiple of 4: a quad ends before it or begins past it)
    __device__ __forceinline__ void four(f32x4& x, const Spot& s, int64_t k, int dk, int64_t kend) const {
        const auto rsrc = buffer_rsrc(base, 0x80000000ll);
        const int plane4 = a->H * a->W * 4;
        uint32_t tap, c, ti, tj;
        fast_divmod((uint32_t)k + dk, a->div_c, tap, c);
        fast_divmod(tap, a->div_kw, ti, tj);
        const bool in = ((unsigned)(s.iy0 + (int)ti) < (unsigned)a->H) &
                        ((unsigned)(s.ix0 + (int)tj) < (unsigned)a->W) & (!PART || k + dk < kend);
        const int at = in ? s.off + (int)c * plane4 + ((int)ti * a->W + (int)tj) * 4 : kOutOfRange;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, at, e * plane4, 0));
    }
};

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS, bool ONE_TAP>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N * KS, 2) void conv_split_kernel(ConvSplitArgs a) {
    using C_ = SplitCfg<BM, BN, BK, WAVES_M, WAVES_N, KS>;
    __shared__ u32x4 smem[2 * C_::STAGE];
    int tm, tn;
    tile_coords(a.g, blockIdx.x, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    SplitOperand<BM, BK, true, C_::NT, C_::UA> oa;
    ConvPixels<BN, BK, C_::NT, C_::UB, ONE_TAP> ob;
    oa.init(a.g.A, a.g.K, m0, a.g.M, -1, threadIdx.x);
    ob.init(a, n0, threadIdx.x);
    split_tile<BM, BN, BK, WAVES_M, WAVES_N, KS, true>(a.g, smem, oa, ob, m0, n0, 0, a.g.K, 0, 0);
}

using ConvKernel = void (*)(ConvSplitArgs);
template <int BM, int BN, int BK, int KS>
ConvKernel conv_form(int channels) {
    return channels % BK ? conv_split_kernel<BM, BN, BK, 2, 2, KS, false>
                         : conv_split_kernel<BM, BN, BK, 2, 2, KS, true>;
}
ConvKernel conv_kernel(int tile, int channels) {
    switch (tile) {
        case S128x128: return conv_form<128, 128, 32, 2>(channels);
        case S64x128: return conv_form<64, 128, 32, 1>(channels);
        case S64x64K: return conv_form<64, 64, 64, 2>(channels);
        default: return conv_form<64, 64, 32, 1>(channels);
    }
}

// ------------------------------------------------------------ weight gradient

// The quad of output pixels at k.
struct QuadAt {
    int live;      // pixels of the quad inside its row (0: past the end)
    int g_off;     // bytes of the quad in a channel plane of the gradient
    int x_off;     // bytes of its window corner in the image's first plane
    int iy0, ix0;  // that corner

    QuadAt() = default;
    __device__ __forceinline__ QuadAt(const ConvSplitArgs& a, int k) {
        const int quad = k >> 2;
        const bool in = quad < a.quads;
        uint32_t row, qx, img, oy;
        fast_divmod((uint32_t)(in ? quad : 0), a.div_rowq, row, qx);
        fast_divmod(row, a.div_oh, img, oy);
        const int ox = 4 * (int)qx;
        live = in ? a.OW - ox : 0;
        g_off = ((int)img * (int)a.g.M * a.OH * a.OW + (int)oy * a.OW + ox) * 4;
        iy0 = (int)oy * a.stride - a.pad_h;
        ix0 = ox * a.stride - a.pad_w;
        x_off = ((int)img * a.C * a.H * a.W + (int)oy * a.stride * a.W + ox * a.stride) * 4;
    }
};

// The two quads that a thread's units of a k-tile cover.
template <int BK>
__device__ __forceinline__ void quad_pos(QuadAt (&p)[2], const ConvSplitArgs& a, int64_t k0, int tid) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
        p[half] = QuadAt(a, (int)k0 + half * (BK / 2) + 4 * (tid % (BK / 8)));
}

// The output gradient [channel][pixel]. QUADS: rows are whole quads.
template <int BM, int BK, int NT, int U, bool QUADS>
struct GradRows {
    static constexpr bool kKC = true, kOnes = false, kMasked = true, kFix = false;
    static constexpr uint32_t ones = 0;
    const ConvSplitArgs* a;
    const QuadAt* pos;  // [2]
    int64_t m0;
    int off[U];

    __device__ __forceinline__ void init(const ConvSplitArgs& args, const QuadAt* p, int64_t m0_,
                                         int tid) {
        a = &args;
        pos = p;
        m0 = m0_;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            int row, q;
            split_pos<BM, BK, true, NT>(i, tid, row, q);
            off[i] = (int)min(m0 + row, a->g.M - 1) * a->OH * a->OW * 4;
        }
    }
    __device__ __forceinline__ void begin(int64_t, int) {}
    __device__ __forceinline__ void fix(f32x4 (&)[2], int) const {}
    // The quad p of the channel at `off`.
    __device__ __forceinline__ void fetch(f32x4& r, int off, const QuadAt& p) const {
        const auto rsrc = buffer_rsrc(a->g.A, 0x80000000ll);
        const int at = off + p.g_off;
        if constexpr (QUADS) {
            r = buffer_load4(rsrc, p.live > 0 ? at : kOutOfRange);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = buffer_load1(rsrc, e < p.live ? at + 4 * e : kOutOfRange);
        }
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&r)[2], int i, int64_t, int64_t, int) const {
#pragma unroll
        for (int half = 0; half < 2; ++half) fetch(r[half], off[i], pos[half]);
    }
    using Spot = int;  // bytes of the row's channel in an image
    __device__ __forceinline__ Spot spot(int row) const {
        return (int)min(m0 + row, a->g.M - 1) * a->OH * a->OW * 4;
    }
    template <bool PART>  // (slices are whole k steps, the last one masked by the quads)
    __device__ __forceinline__ void four(f32x4& x, const Spot& s, int64_t k, int dk, int64_t) const {
        fetch(x, s, QuadAt(*a, (int)k + dk));
    }
};

// The im2col matrix [c * taps + tap][pixel], and the column of ones after it.
// NEAR: whole quads of a stride-1 layer with at most one column of padding: a
// quad's four window pixels are one 128-bit load (a quarter of the load
// instructions). Where the window's first or last pixel is outside the image
// the load moves one pixel in, and `settle` moves the values back.
template <int BN, int BK, int NT, int U, bool NEAR>
struct WindowRows {
    static constexpr bool kKC = true, kOnes = true, kMasked = true, kFix = NEAR;
    const ConvSplitArgs* a;
    QuadAt pos[2];
    const float* base;  // the image, one padding corner before its start
    int64_t n0;
    int off[U], ti[U], tj[U];
    uint32_t moved[U];  // NEAR: bits 2 half (left), 2 half + 1 (right) of each unit in flight
    uint32_t ones = 0;

    __device__ __forceinline__ int64_t columns() const { return (int64_t)a->C * a->taps; }
    __device__ __forceinline__ void init(const ConvSplitArgs& args, int64_t n0_, int tid) {
        a = &args;
        n0 = n0_;
        base = a->g.B - (a->pad_h * a->W + a->pad_w);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            int row, q;
            split_pos<BN, BK, true, NT>(i, tid, row, q);
            ones |= (uint32_t)(n0 + row == columns()) << i;
            uint32_t c, tap, y, x;
            fast_divmod((uint32_t)min(n0 + row, columns() - 1), a->div_taps, c, tap);
            fast_divmod(tap, a->div_kw, y, x);
            ti[i] = (int)y;
            tj[i] = (int)x;
            off[i] = ((int)c * a->H * a->W + (int)y * a->W + (int)x) * 4;
        }
    }
    __device__ __forceinline__ void begin(int64_t k0, int tid) { quad_pos<BK>(pos, *a, k0, tid); }
    // The window pixels of quad p at tap (ty, tx), `off` bytes from its corner;
    // returns what `settle` has to know.
    __device__ __forceinline__ uint32_t fetch(f32x4& r, int off, int ty, int tx, const QuadAt& p) const {
        const auto rsrc = buffer_rsrc(base, 0x80000000ll);
        const bool row_in = (unsigned)(p.iy0 + ty) < (unsigned)a->H;
        if constexpr (NEAR) {
            const int ix = p.ix0 + tx;
            const bool in = row_in & (p.live > 0);
            const bool left = ix < 0, right = ix + 3 >= a->W;
            const int at = off + p.x_off + (left ? 4 : 0) - (right ? 4 : 0);
            r = buffer_load4(rsrc, in ? at : kOutOfRange);
            return (uint32_t)left | (uint32_t)right << 1;
        } else {
            const int at = off + p.x_off, ix = row_in ? p.ix0 + tx : -(1 << 28);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool ok = ((unsigned)(ix + e * a->stride) < (unsigned)a->W) & (e < p.live);
                r[e] = buffer_load1(rsrc, ok ? at + 4 * e * a->stride : kOutOfRange);
            }
            return 0;
        }
    }
    static __device__ __forceinline__ void settle(f32x4& r, uint32_t moved) {
        if constexpr (NEAR) {
            const bool left = moved & 1u, right = moved & 2u;
            const f32x4 v = r;
            r = f32x4{right ? v[1] : (left ? 0.0f : v[0]), right ? v[2] : (left ? v[0] : v[1]),
                      right ? v[3] : (left ? v[1] : v[2]), right ? 0.0f : (left ? v[2] : v[3])};
        }
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&r)[2], int i, int64_t, int64_t, int) {
        moved[i] = 0;
#pragma unroll
        for (int half = 0; half < 2; ++half)
            moved[i] |= fetch(r[half], off[i], ti[i], tj[i], pos[half]) << (2 * half);
    }
    __device__ __forceinline__ void fix(f32x4 (&r)[2], int i) const {
#pragma unroll
        for (int half = 0; half < 2; ++half) settle(r[half], moved[i] >> (2 * half));
    }
    struct Spot {
        int off, ty, tx;  // bytes of the channel's tap in an image, and the tap
        bool ones;
    };
    __device__ __forceinline__ Spot spot(int col) const {  // (columns past the ones are not stored)
        uint32_t c, tap, ty, tx;
        fast_divmod((uint32_t)min(n0 + col, columns() - 1), a->div_taps, c, tap);
        fast_divmod(tap, a->div_kw, ty, tx);
        return Spot{((int)c * a->H * a->W + (int)ty * a->W + (int)tx) * 4, (int)ty, (int)tx,
                    n0 + col == columns()};
    }
    template <bool PART>
    __device__ __forceinline__ void four(f32x4& x, const Spot& s, int64_t k, int dk, int64_t) const {
        settle(x, fetch(x, s.off, s.ty, s.tx, QuadAt(*a, (int)k + dk)));
        if (s.ones) x = f32x4{1.0f, 1.0f, 1.0f, 1.0f};
    }
};

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS, bool QUADS, bool NEAR>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N * KS, 2) void conv_split_wgrad_kernel(
    ConvSplitArgs a) {
    using C_ = SplitCfg<BM, BN, BK, WAVES_M, WAVES_N, KS>;
    __shared__ u32x4 smem[2 * C_::STAGE];
    int bid = blockIdx.x, slice = blockIdx.y, tm, tn;
    if (gridDim.y > 1 && (gridDim.x & 7) != 0)
        split_coords(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x, gridDim.y, bid, slice);
    tile_coords(a.g, bid, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int64_t kbeg = (int64_t)slice * a.g.k_per_slice;
    const int64_t kend = min(a.g.K, kbeg + a.g.k_per_slice);
    GradRows<BM, BK, C_::NT, C_::UA, QUADS> oa;
    WindowRows<BN, BK, C_::NT, C_::UB, NEAR> ob;
    ob.init(a, n0, threadIdx.x);
    oa.init(a, ob.pos, m0, threadIdx.x);
    // (A's units are loaded first, from the positions B's begin finds: the
    // tile's begin calls come before any load)
    split_tile<BM, BN, BK, WAVES_M, WAVES_N, KS, true>(a.g, smem, oa, ob, m0, n0, kbeg, kend, slice,
                                                       0);
}

// dw[m][n] = sum over slices of part[slice][m][n] + beta * dw, n < cols, and
// db[m] from column cols. A workgroup is groups of WAVES waves, each group 64
// outputs and a run of slices a wave, the runs added in order: with a thread per
// output, a small layer's few thousand outputs over 256 slices were one long
// chain of loads (M 32, 145 columns: 12.4 us, now 5). No more waves than slices:
// of 16, the 5x5 weight gradient of 256 -> 256 channels over a 7x7 image, 1.6
// million outputs of one slice, kept 15 idle and took 62 us, with one 22. WAVES
// is the kernel's own, so that a group's runs are read from LDS together: with a
// loop of unknown length 110,720 outputs of 16 slices took 8.9 us, now 6.6.
constexpr int kSumWaves = 16;
constexpr int sum_threads(int waves) { return waves < 4 ? 256 : 64 * waves; }
template <int WAVES>
__global__ __launch_bounds__(sum_threads(WAVES)) void conv_split_sum_kernel(
    float* dw, float* db, const float* part, int slices, int M, int cols, float beta, FastDiv div_n) {
    constexpr int kGroups = sum_threads(WAVES) / (64 * WAVES);
    __shared__ float red[kGroups * WAVES][64];
    const int total = M * (cols + 1), tx = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6, ty = wave % WAVES, group = wave / WAVES;
    const int e = (blockIdx.x * kGroups + group) * 64 + tx;
    const int per = (slices + WAVES - 1) / WAVES;
    const int s0 = ty * per, s1 = min(slices, s0 + per);
    const float* src = part + min(e, total - 1);
    float v = 0.0f;
    if (per <= 2) {  // uniform; short runs without the loads past their end
        for (int s = s0; s < s1; ++s) v += src[(int64_t)s * total];
    } else {
        for (int s = s0; s < s1; s += 16) {
            float x[16];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = src[(int64_t)min(s + j, s1 - 1) * total];
            if (s + 8 < s1) {
#pragma unroll
                for (int j = 8; j < 16; ++j) x[j] = src[(int64_t)min(s + j, s1 - 1) * total];
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) v += s + j < s1 ? x[j] : 0.0f;
        }
    }
    red[wave][tx] = v;
    __syncthreads();
    if (ty || e >= total) return;
#pragma unroll
    for (int y = 1; y < WAVES; ++y) v += red[wave + y][tx];
    uint32_t m, n;
    fast_divmod((uint32_t)e, div_n, m, n);
    float* dst = (int)n < cols ? dw + (int64_t)m * cols + n : (db ? db + m : nullptr);
    if (dst) *dst = beta != 0.0f ? v + beta * *dst : v;
}

using SumKernel = void (*)(float*, float*, const float*, int, int, int, float, FastDiv);
SumKernel sum_kernel(int waves) {
    switch (waves) {
        case 1: return conv_split_sum_kernel<1>;
        case 2: return conv_split_sum_kernel<2>;
        case 4: return conv_split_sum_kernel<4>;
        case 8: return conv_split_sum_kernel<8>;
        default: return conv_split_sum_kernel<kSumWaves>;
    }
}

using WgradKernel = void (*)(ConvSplitArgs);

template <int BM, int BN, int WAVES_M, int KS>
WgradKernel wgrad_form(int form) {
    switch (form) {
        case 0: return conv_split_wgrad_kernel<BM, BN, 32, WAVES_M, 2, KS, false, false>;
        case 1: return conv_split_wgrad_kernel<BM, BN, 32, WAVES_M, 2, KS, true, false>;
        default: return conv_split_wgrad_kernel<BM, BN, 32, WAVES_M, 2, KS, true, true>;
    }
}
// Tiles of the weight gradient: `fit` workgroups share a CU (by LDS). Staging
// a column operand unit costs more than its products, so a tile is as wide as
// the columns allow, but for at most 32 rows: there half of a 64-row tile's
// products are padding, and past 128 columns 64-wide tiles also pad less and
// leave four workgroups a CU to cover each other's gathering. 64x128 against
// 32x64 (us, with the sum): 16->32 3x3 32 x 64^2 42.0 / 33.5 (145 columns), 16 x
// 32->32 64^2 35.4 / 28.4, 16 x 128->32 56^2 70.4 / 57.8, 1x1 128->32 32 x 32^2
// 21.5 / 17.9; one wide tile of columns stays ahead: 8->32 64 x 32^2 (73
// columns) 19.8 / 20.8, 3->32 32 x 64^2 (28) 21.3 / 23.3.
struct WgradTile {
    int bm, bn, threads, fit;
    WgradKernel kernel;
};
WgradTile wgrad_tile(int64_t M, int64_t N, int form) {
    if (M <= 32 && N > 128) return {32, 64, 128, 4, wgrad_form<32, 64, 1, 1>(form)};
    if (N <= 64) return {64, 64, 256, 2, wgrad_form<64, 64, 2, 1>(form)};
    if (M <= 64) return {64, 128, 256, 2, wgrad_form<64, 128, 2, 1>(form)};
    return {128, 128, 512, 1, wgrad_form<128, 128, 2, 2>(form)};
}

}  // namespace

int split_conv(const SlabConv& s) {
    if (!split_conv_takes(s)) return kSlabUnsupported;
    const int64_t taps = (int64_t)s.kh * s.kw, P = (int64_t)s.OH * s.OW, pixels = s.N * P;
    ConvSplitArgs a{};
    GemmArgs& g = a.g;
    g.B = s.x;
    g.C = s.out;
    g.bias = s.bias;
    g.M = g.mrows = s.M;
    g.N = pixels;
    g.K = taps * s.C;
    g.ldc = g.N;
    g.beta = s.beta;
    g.epi = s.bias ? NRS_EPI_BIAS_ROW : NRS_EPI_NONE;
    g.nchw_P = P;
    g.div_nchw = make_fastdiv((uint32_t)P);
    g.group_m = 8;
    a.C = s.C;
    a.H = s.H;
    a.W = s.W;
    a.taps = (int)taps;
    a.kw = s.kw;
    a.stride = s.stride;
    a.pad_h = s.pad_h;
    a.pad_w = s.pad_w;
    a.OH = s.OH;
    a.OW = s.OW;
    a.div_c = make_fastdiv((uint32_t)s.C);
    a.div_kw = make_fastdiv((uint32_t)s.kw);
    a.div_p = make_fastdiv((uint32_t)P);
    a.div_ow = make_fastdiv((uint32_t)s.OW);
    const int tile = split_conv_tile(s, num_cus());
    const int bm = tile == S128x128 ? 128 : 64, bn = tile == S64x64K || tile == S64x64 ? 64 : 128;
    g.tiles_m = (int)cdiv(s.M, bm);
    g.tiles_n = (int)cdiv(pixels, bn);
    if ((int64_t)g.tiles_m * g.tiles_n > INT32_MAX) return kSlabUnsupported;
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n));
    const int wn = (int)(s.M * g.K);
    float* packed = workspace(sizeof(float) * (size_t)wn, 4);
    if (!packed) return NRS_ERR_ALLOC;
    g.A = packed;
    hipLaunchKernelGGL(conv_split_weights_kernel,
                       dim3((unsigned)std::min<int64_t>(cdiv(wn, 256), 4 * (int64_t)num_cus())),
                       dim3(256), 0, stream(), packed, s.w, s.M, s.C, (int)taps, s.flip ? 1 : 0,
                       a.div_c, make_fastdiv((uint32_t)taps));
    NRS_LAUNCH_CHECK("conv2d (split, weights)");
    const bool threads512 = tile == S128x128 || tile == S64x64K;
    hipLaunchKernelGGL(conv_kernel(tile, s.C), grid, dim3(threads512 ? 512 : 256), 0, stream(), a);
    NRS_LAUNCH_CHECK("conv2d (split)");
    return NRS_OK;
}

int split_wgrad(const SlabWgrad& s) {
    const int64_t taps = (int64_t)s.kh * s.kw, cols = s.C * taps, row_q = cdiv(s.OW, 4);
    const int64_t quads = s.N * s.OH * row_q;
    const int64_t in_bytes = s.N * s.C * s.H * s.W * 4 + ((int64_t)s.pad * s.W + s.pad) * 4;
    const int64_t grad_bytes = s.N * s.M * s.OH * s.OW * 4;
    if (quads > (1 << 28) || in_bytes > 0x7fffffffll || grad_bytes > 0x7fffffffll || cols > (1 << 24) ||
        (int64_t)s.M * (cols + 1) > (1 << 28))
        return kSlabUnsupported;
    ConvSplitArgs a{};
    GemmArgs& g = a.g;
    g.A = s.g;
    g.B = s.x;
    g.M = g.mrows = s.M;
    g.N = cols + 1;
    g.K = cdiv(quads * 4, 32) * 32;
    g.group_m = 8;
    a.C = s.C;
    a.H = s.H;
    a.W = s.W;
    a.taps = (int)taps;
    a.kw = s.kw;
    a.stride = s.stride;
    a.pad_h = a.pad_w = s.pad;
    a.OH = s.OH;
    a.OW = s.OW;
    a.quads = (int)quads;
    a.div_kw = make_fastdiv((uint32_t)s.kw);
    a.div_taps = make_fastdiv((uint32_t)taps);
    a.div_rowq = make_fastdiv((uint32_t)row_q);
    a.div_oh = make_fastdiv((uint32_t)s.OH);
    const int form = s.OW % 4 ? 0 : (s.stride == 1 && s.pad <= 1 && s.W >= 4 ? 2 : 1);
    const WgradTile t = wgrad_tile(s.M, g.N, form);
    g.tiles_m = (int)cdiv(s.M, t.bm);
    g.tiles_n = (int)cdiv(g.N, t.bn);
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n, ksteps = g.K / 32;
    // One round of workgroups (one 128x128 tile fits a CU, two of the others),
    // at most 256 slices, and of a short reduction as many as balance a slice's
    // k steps (1.1 us each) with adding a slice (0.03 us and 1 us a million
    // outputs): 16->32 8 x 8x8, 16 steps, 13.0 us with 4 steps a slice, 9.4 with
    // 1; 64 x 14x14, 392 steps, 15.4 with 4, 17.2 with 2; 32->48 8 x 30x30, 240
    // steps, 16.6 with 4, 19.3 with 2.
    const int64_t round = t.fit * (int64_t)num_cus();
    const double add = 0.03 + 1e-6 * (double)(s.M * g.N), step = 1.1;
    const int64_t least = std::max<int64_t>(1, std::llround(std::sqrt((double)ksteps * add / step)));
    int64_t slices = std::max<int64_t>(1, std::min({round / tiles, cdiv(ksteps, least), (int64_t)256}));
    g.k_per_slice = cdiv(ksteps, slices) * 32;
    slices = cdiv(g.K, g.k_per_slice);
    g.partial = workspace(sizeof(float) * (size_t)(slices * s.M * g.N), 3);
    if (!g.partial) return NRS_ERR_ALLOC;
    const dim3 grid((unsigned)tiles, (unsigned)slices);
    hipLaunchKernelGGL(t.kernel, grid, dim3(t.threads), 0, stream(), a);
    NRS_LAUNCH_CHECK("conv2d weight gradient (split)");
    const int64_t total = s.M * g.N;
    int waves = 1;
    while (waves < kSumWaves && waves < slices) waves *= 2;
    const int threads = sum_threads(waves);
    hipLaunchKernelGGL(sum_kernel(waves), dim3((unsigned)cdiv(total, threads / waves)), dim3(threads), 0,
                       stream(), s.dw, s.db, g.partial, (int)slices, s.M, (int)cols, s.beta,
                       make_fastdiv((uint32_t)g.N));
    NRS_LAUNCH_CHECK("conv2d weight gradient (split, sum)");
    return NRS_OK;
}

}  // namespace nrs
