// Which products the split GEMM (gemm_split.hpp) takes, on which tile and in
// how many K slices. Host only and free of HIP, so that a CPU test can ask.
#pragma once

#include <algorithm>
#include <cstdint>

#include "nrs_hip.h"

namespace nrs {

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Tiles of the split GEMM.
enum SplitTile { S256x256 = 0, S128x128, S64x128, S64x64K, S64x64, S_COUNT };

// What a k step of 32 costs a workgroup (us:
// `alone` on its CU, `shared` with others there) and what it costs besides
// (filling the pipeline, the epilogue), fitted to whole grids of
// 1024^2, 2048^2 and 4096^2 over K = 32 .. 512, e.g. (us)
//   4096^2 over 64 / 512   256x256 24 / 90    128x128 32 / 117   64x128 28 / 134
//   2048^2 over 64 / 512   128x128 10 / 31    64x128 8.9 / 32    64x64 10 / 35
//   1024^2 over 64 / 512   64x64K 5.1 / 11.3  64x64 5.2 / 13.6   128x128 7.5 / 21
// (a 256x128 tile with second accumulators takes 660 us for 4096^3, the
// 256x256 one 590). The two costs of the narrow tiles for dense operands are
// fitted to 65 ragged and batched products as well, where three 64x64
// workgroups on a CU cover each other's partial last k step (64x128 / 64x64, us):
//   32 x 276x128 over 40 8.2 / 7.0    723x1626 over 126 10.2 / 8.7
//   85 x 74x128 over 393 17.2 / 15.9  687x2393 over 1263 43.2 / 41.3
//   162 x 315x89 over 80 21.9 / 23.8  1947x1635 over 92 12.5 / 13.5
// (the choice is 0.9% from the best tile in the mean, 2.2% with the whole
// grids' costs). Gathered operands keep those: staging a wide tile costs less.
struct SplitCost {
    double alone, shared, fixed;
};
struct SplitShape {
    int bm, bn, bk, threads;
    SplitCost dense, gathered;
};
constexpr SplitShape kSplitShapes[S_COUNT] = {
    {256, 256, 16, 512, {4.55, 4.55, 12.5}, {4.55, 4.55, 12.5}},
    {128, 128, 32, 512, {1.5, 1.5, 4.5}, {1.5, 1.5, 4.5}},
    {64, 128, 32, 256, {0.93, 0.9, 1.75}, {0.93, 0.9, 1.6}},
    {64, 64, 64, 512, {0.45, 0.5, 1.9}, {0.45, 0.5, 1.9}},
    {64, 64, 32, 256, {0.61, 0.4, 1.0}, {0.61, 0.456, 1.25}},
};

// A dense product: C[M][N] over K, `batch` of them, with or without a row of
// sums; `split_k` if it may be split over K, `wide` if the f32 kernels would
// load it in 128 bits (aligned rows of whole float4s).
struct GemmSize {
    int layout;
    int64_t M, N, K, batch;
    bool sum_row = false, split_k = true, wide = false;
    int64_t lda() const { return layout == NRS_TN ? M : K; }
    int64_t ldb() const { return layout == NRS_NT ? K : N; }
};

// Whether the 32-bit byte offsets of a staged tile hold: within the rows of a
// tile of an operand contiguous in k, within a k step of another. (64-row tiles
// reach rows of 8.5 million floats. A wide layer of 512 x 2.5 million over 128
// takes 2275 us on them and 3324 on the f32 kernel.)
inline bool split_addressable(const GemmSize& s, int tile) {
    const SplitShape& t = kSplitShapes[tile];
    const auto reach = [&](bool contiguous_k, int64_t rows, int64_t ld) {
        return 4 * (contiguous_k ? (rows - 1) * ld + t.bk : (t.bk - 1) * ld + rows);
    };
    return reach(s.layout != NRS_TN, t.bm, s.lda()) <= INT32_MAX &&
           reach(s.layout == NRS_NT, t.bn, s.ldb()) <= INT32_MAX;
}

// The group kernel (64x64x32 tiles) takes products of any size it can address
// (a row of ones is built for TN only).
inline bool group_takes(const GemmSize& s) {
    return s.K > 0 && split_addressable(s, S64x64) && (!s.sum_row || s.layout == NRS_TN);
}
inline bool any_tile_addresses(const GemmSize& s) {
    bool any = false;
    for (int t = 0; t < S_COUNT; ++t) any = any || split_addressable(s, t);
    return any && s.K > 0 && (!s.sum_row || s.layout == NRS_TN);
}

// Whether every product of nrs_matmul_shared_lhs_backward fits the group
// kernel: dx (+)= g . W^T and dW = x^T . g.
inline bool shared_lhs_fits(int64_t rows, int64_t inner, int64_t cols) {
    return group_takes(GemmSize{NRS_NT, rows, inner, cols, 1}) &&
           group_takes(GemmSize{NRS_TN, inner, cols, rows, 1});
}

// The tile of the least estimated time for an unsplit product, and that time
// in us. `gathered`: a convolution's operand; `dense`: a dense product, whose
// tile must address it.
inline int cheapest_split_tile(int64_t M, int64_t N, int64_t K, int64_t batch, bool gathered,
                               int cus, double* time = nullptr, const GemmSize* dense = nullptr) {
    int best = S64x64;
    double least = 1e30;
    for (int t = 0; t < S_COUNT; ++t) {
        const SplitShape& s = kSplitShapes[t];
        const SplitCost& cost = gathered ? s.gathered : s.dense;
        if (dense && !split_addressable(*dense, t)) continue;
        const int64_t per_cu = cdiv(cdiv(M, s.bm) * cdiv(N, s.bn) * batch, (int64_t)cus);
        const double steps = (double)(cdiv(K, s.bk) * s.bk) / 32.0;
        const double est =
            (double)per_cu * (steps * (per_cu > 1 ? cost.shared : cost.alone) + cost.fixed);
        if (est < least) {
            least = est;
            best = t;
        }
    }
    if (time) *time = least;
    return best;
}

// Whether a product of a short reduction is ahead on the f32 kernel's 64x64 tile:
// over at most one of its k steps with 128-bit loads, and up to two where the
// split's second step is a partial one of an operand contiguous in k, which it
// loads value by value. Both ways over 38000 products, split against f32 (us):
//   100 x 50000 over 32 NN 15.9 / 12.5   20860 x 128 over 52 NT 11.0 / 8.5
//   23 x 638x404 over 24 NT 15.0 / 11.9  over 64 64x64 tiles 0.99x
//   without 128-bit loads over 32 .. 64 0.70x to 0.97x
//   256x256 tiles over 32 1.08x, of whole tiles 0.98x, over 16 0.92x
inline bool f32_ahead(const GemmSize& s, int cus) {
    if (!s.wide || s.K >= 64) return false;
    const bool big = cheapest_split_tile(s.M, s.N, s.K, s.batch, false, cus, nullptr, &s) == S256x256;
    if (big) return s.K > 16 && s.K <= 32 && (s.M % 256 || s.N % 256);
    return s.K <= 32 || s.layout != NRS_TN;
}

// The split GEMM takes dense products of more than 32 rows and columns. The f32
// tiles keep gathered operands, outputs of at most 32 rows or columns
// (padding would leave the matrix cores nothing to gain), short reductions where
// they are ahead and those under a k step into few tiles (1024 x 1024 over 16: 4.4
// us against 4.7; with four tiles a CU the split tiles win again without 128-bit
// loads).
inline bool split_takes(const GemmSize& s, int cus) {
    return s.M > 32 && s.N > 32 && any_tile_addresses(s) && !f32_ahead(s, cus) &&
           (s.K >= 32 || cdiv(s.M, 64) * cdiv(s.N, 64) * s.batch >= 4 * (int64_t)cus);
}

struct SplitPlan {
    int tile, slices;
    int64_t k_per_slice;
};

// Outputs of few 64x64 tiles over a long reduction are split over K, into
// about three workgroups a CU, others take one tile's time.
inline SplitPlan plan_split(const GemmSize& s, int cus) {
    const int64_t M = s.M + (s.sum_row ? 1 : 0), N = s.N, K = s.K;
    const int64_t t64 = cdiv(M, 64) * cdiv(N, 64) * s.batch;
    if (s.split_k && s.batch == 1 && split_addressable(s, S64x64) && t64 < cus && (2 * t64 <= cus || K >= 2048) && K >= 256) {
        const int64_t want = std::min<int64_t>(256, cdiv(3 * (int64_t)cus, t64));
        const int64_t max_by_k = std::max<int64_t>(1, K / ((t64 >= 16 ? 8 : 2) * 32));
        const int64_t slices = std::max<int64_t>(1, std::min(want, max_by_k));
        const int64_t kps = cdiv(cdiv(K, slices), 32) * 32;
        return SplitPlan{S64x64, (int)cdiv(K, kps), kps};
    }
    const int tile = cheapest_split_tile(M, N, K, s.batch, false, cus, nullptr, &s);
    const int bk = kSplitShapes[tile].bk;
    return SplitPlan{tile, 1, cdiv(K, bk) * bk};
}

}  // namespace nrs
