// Kernels of the split GEMM (gemm_split.hpp): one instance per tile and layout.
#include "gemm_split.hpp"

namespace nrs {
namespace {

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS, bool TWO = true>
SplitKernel pick(int layout) {
    switch (layout) {
        case NRS_NN: return gemm_split_kernel<BM, BN, BK, WAVES_M, WAVES_N, KS, TWO, true, false>;
        case NRS_NT: return gemm_split_kernel<BM, BN, BK, WAVES_M, WAVES_N, KS, TWO, true, true>;
        default: return gemm_split_kernel<BM, BN, BK, WAVES_M, WAVES_N, KS, TWO, false, false>;
    }
}

}  // namespace

SplitKernel split_kernel(int tile, int layout) {
    switch (tile) {
        case S256x256: return pick<256, 256, 16, 2, 4, 1, false>(layout);
        case S128x128: return pick<128, 128, 32, 2, 2, 2>(layout);
        case S64x128: return pick<64, 128, 32, 2, 2, 1>(layout);
        case S64x64K: return pick<64, 64, 64, 2, 2, 2>(layout);
        default: return pick<64, 64, 32, 2, 2, 1>(layout);
    }
}

SplitGroupKernel split_group_kernel() { return gemm_split_group_kernel<64, 64, 32, 2, 2>; }

}  // namespace nrs
