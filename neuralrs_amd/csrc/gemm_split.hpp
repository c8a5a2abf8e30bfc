// Device side of the split GEMM: f32 products on the bf16 matrix cores.
//
// The f32 matrix instructions of gfx950 run at 157 TFLOP/s, the bf16 ones at
// 2.3 PFLOP/s. A float is the exact sum of three bf16 pieces of 8 significand
// bits each,
//   x = x0 + x1 + x2,  x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1,
// so a product of two floats is the sum of nine products of pieces, each of
// them exact in f32 (Henry, Tang and Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations", ARITH
// 2019). The six with i + j <= 2 are accumulated in f32 by
// v_mfma_f32_32x32x16_bf16. With pieces rounded to nearest |x1| <= 2^-8 |x| and
// |x2| <= 2^-17 |x|, so the other three are at most 2^-24 of the product, as
// much as rounding it once (0.84 of that at most over two million random
// pairs), and have no common sign: a sum of one or two terms can be a unit
// further off than f32 multiply-adds, sums of many are closer (below).
// An instruction adds its 16 products in two halves of 8. In each, bits of the
// products below 2^-24 of the largest are dropped, and the accumulator is
// rounded once: twice for 16 products, the f32 instructions once a product.
// TWO: the products of first pieces have an accumulator of their own and the
// other five share a second one, at most 2^-7 of its size, so the large sum is rounded
// K / 8 times. Without (the 256x256 tile, whose second accumulators would not
// fit the registers) it is rounded 6 K / 8 times. Error against 64 bits of one
// 32x32 block, f32 instructions / one accumulator / two:
//   uniform values   K = 256  2.8e-7 / 2.3e-7 / 0.8e-7   4096  1.2e-6 / 1.0e-6 / 3.9e-7
//   normal values    K = 256  3.0e-7 / 2.4e-7 / 1.0e-7   4096  1.1e-6 / 1.0e-6 / 4.1e-7
//
// The split is exact for every float of magnitude 2^-110 and more (below,
// x2 may need bits under bf16's smallest denormal) whose x0 is finite. Both
// exceptions are seen and computed again on the f32 instructions, 32x32 blocks
// of C at a time, from global memory (f32_block):
//  * staging keeps, for every row a thread stages units of, the OR of the bits
//    of its x2s that their bf16 form drops. How much those bits matter depends
//    on what they would have met (2^-134 of a row by 2^120 of a column is a
//    normal result), so the results of every row of A and column of B that
//    dropped any are replaced, whatever their size;
//  * results that are infinite or NaN (an infinite or NaN input, a value that
//    rounds past bf16's range, or a true overflow) are replaced.
// Which instructions a result comes from thus depends on its own row of A and
// column of B alone: a sample's bits don't change with the others of its batch.
//
// A workgroup of WAVES_M x WAVES_N waves owns a BM x BN block of C. Operand
// tiles of BK k values are loaded to registers one k-tile ahead, split, and
// stored as three bf16 planes in one of two LDS buffers, in units of 8 k
// values of one row (16 bytes, one lane's MFMA operand): the unit of row r,
// unit index q lies at ((r / 32) * (BK / 8) + q) * 32 + (r % 32 ^ swizzle(q)),
// so operand reads are contiguous per wave and the staging stores of
// neighbouring lanes (rows x units) hit distinct banks. Unit q holds
// k = 4q .. 4q+3 and BK/2 + 4q .. BK/2 + 4q + 3 of the tile, the same for A
// and B: a row's lanes then load whole 64- or 128-byte segments when the
// operand is contiguous in k. Loads are 4-byte aligned 128-bit buffer loads
// there, and dword loads of 64 neighbouring columns otherwise, so any leading
// dimension and alignment takes the same path.
#pragma once

#include <cfloat>

#include "gemm_kernel.hpp"

namespace nrs {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The split of the 8 floats of a unit in kSplitSteps steps of four independent
// vector instructions each. A dependent instruction waits ten cycles on
// gfx950, an independent one five: the steps are dealt out between matrix
// instructions (32 cycles), which up to four of them a matrix instruction
// leave at full rate (a remainder by v_dot2_f32_bf16, one instruction in place
// of two, does not: dot products and matrix products exclude each other, and
// two a matrix instruction halve its rate). The empty asm pins each step's
// place. Bits of x2 that its bf16 form drops go to `sticky` (low 16 bits).
constexpr int kSplitSteps = 12;

struct SplitState {
    float a[4], b[4];       // remainders of the even and the odd floats
    uint32_t lo[4], hi[4];  // a piece of each, as floats
    u32x4 piece[3];         // packed pieces: even floats in the low halves

    template <int n>
    __device__ __forceinline__ void step(const f32x4 (&v)[2], uint32_t& sticky, bool one) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (n == 0) {
                a[i] = one ? 1.0f : v[i / 2][i % 2 * 2];
                b[i] = one ? 1.0f : v[i / 2][i % 2 * 2 + 1];
            }
            if constexpr (n == 0 || n == 5) {
                uint32_t p = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a[i], (__bf16)b[i]});
                asm volatile("" : "+v"(p));
                piece[n / 5][i] = p;
            } else if constexpr (n == 1 || n == 6) {
                lo[i] = piece[n / 5][i] << 16;
                asm volatile("" : "+v"(lo[i]));
            } else if constexpr (n == 2 || n == 7) {
                hi[i] = piece[n / 5][i] & 0xffff0000u;
                asm volatile("" : "+v"(hi[i]));
            } else if constexpr (n == 3 || n == 8) {
                a[i] -= __builtin_bit_cast(float, lo[i]);
                asm volatile("" : "+v"(a[i]));
            } else if constexpr (n == 4 || n == 9) {
                b[i] -= __builtin_bit_cast(float, hi[i]);
                asm volatile("" : "+v"(b[i]));
            } else if constexpr (n == 10) {
                uint32_t p = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b[i]),
                                                   __builtin_bit_cast(uint32_t, a[i]), 0x07060302u);
                asm volatile("" : "+v"(p));
                piece[2][i] = p;
            } else {
                sticky |= __builtin_bit_cast(uint32_t, a[i]) | __builtin_bit_cast(uint32_t, b[i]);
            }
        }
        if constexpr (n == kSplitSteps - 1) asm volatile("" : "+v"(sticky));
    }
};

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS>
struct SplitCfg {
    static constexpr int NT = 64 * WAVES_M * WAVES_N * KS;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    static constexpr int FM = WM / 32, FN = WN / 32;
    static constexpr int Q = BK / 8;  // units of a row
    static constexpr int UA = BM * Q / NT, UB = BN * Q / NT;  // units a thread stages
    static constexpr int PLANE_A = BM * Q, PLANE_B = BN * Q;  // units of a plane
    static constexpr int STAGE = 3 * (PLANE_A + PLANE_B);     // units of a buffer
    static_assert(BK == 16 || BK == 32 || BK == 64, "swizzle");
    static_assert(BK % (16 * KS) == 0, "k-split wave sets");
    static_assert(UA * NT == BM * Q && UB * NT == BN * Q && UA >= 1 && UB >= 1, "unit split");
    static_assert(FM >= 1 && FN >= 1 && FM * 32 * WAVES_M == BM && FN * 32 * WAVES_N == BN, "waves");
    static_assert(2 * STAGE * 16 <= 160 * 1024, "LDS budget");
};

// LDS unit index of (row, q) within a plane. The swizzle sends the 8 (and 16)
// units of neighbouring lanes, Q of each row, to distinct 16-byte columns of a
// 128- (256-) byte line: (q ^ 2q) * 8 / Q differs between units of a row in the
// bits just above those of the rows, at either width.
template <int BK>
__device__ __forceinline__ int split_unit(int row, int q) {
    constexpr int Q = BK / 8;
    return ((row >> 5) * Q + q) * 32 + ((row & 31) ^ ((q ^ (q << 1)) * (8 / Q)));
}

// Row (of BMN) and unit of a thread's unit i: lanes run along the rows when
// the operand is contiguous there, else along the units of a row.
template <int BMN, int BK, bool KC, int NT>
__device__ __forceinline__ void split_pos(int i, int tid, int& row, int& q) {
    constexpr int Q = BK / 8;
    const int u = tid + i * NT;
    if (KC) {
        row = u / Q;
        q = u % Q;
    } else {
        row = u % BMN;
        q = u / BMN;
    }
}

// One operand of a workgroup's tile: where its k-tiles start, and the byte
// offset of each of the thread's units there (rows past the operand read its
// last row: their results are not stored). The k-tile's address is in the
// buffer's base, so offsets stay below 256 rows of the operand.
// (What split_tile asks of an operand: kKC, the order of its units over the
// threads; kOnes and `ones`, bit i set where unit i is all ones; kMasked, true
// if load<false> reads zero past the end of k; begin, called before the first
// unit of a k-tile is loaded; load; spot and four, a row and 4 k values of it
// as f32_block takes them, k a multiple of 4; and kFix, of a column operand whose
// loaded units go through fix before they are split.)
template <int BMN, int BK, bool KC, int NT, int U, bool ONES = false>
struct SplitOperand {
    static constexpr bool kKC = KC, kOnes = ONES, kMasked = false, kFix = false;
    const float* base;  // the tile's first row (column) at k = 0
    int64_t ld;
    int off[U];
    int last;  // last row of the operand in the tile
    uint32_t ones = 0;
    int one_row = -1;

    // `one`: the operand row made of ones (-1: none).
    __device__ __forceinline__ void init(const float* X, int64_t ld_, int64_t mn0, int64_t MN,
                                         int64_t one, int tid) {
        ld = ld_;
        const int64_t first = min(mn0, MN - 1);
        base = X + (KC ? first * ld : first);
        last = (int)min((int64_t)(BMN - 1), MN - 1 - first);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            int row, q;
            split_pos<BMN, BK, KC, NT>(i, tid, row, q);
            const int mn = min(row, last);
            off[i] = 4 * (KC ? mn * (int)ld + 4 * q : mn + 4 * q * (int)ld);
            if constexpr (ONES) ones |= (uint32_t)(mn0 + row == one) << i;
        }
        if constexpr (ONES) one_row = one >= 0 ? (int)(one - mn0) : -1;
    }

    __device__ __forceinline__ void begin(int64_t, int) {}
    __device__ __forceinline__ void fix(f32x4 (&)[2], int) const {}

    struct Spot {
        int off;  // bytes of the row at k = 0 of the tile
        bool one;
    };
    __device__ __forceinline__ Spot spot(int row) const {
        const int r = min(row, last);
        return Spot{4 * (KC ? r * (int)ld : r), ONES && row == one_row};
    }
    // Elements k + dk .. k + dk + 3 of a row, k uniform; with PART, zero at or
    // past kend.
    template <bool PART>
    __device__ __forceinline__ void four(f32x4& x, const Spot& s, int64_t k, int dk, int64_t kend) const {
        const auto rsrc = at_k(k);
        const int off = s.off + 4 * dk * (KC ? 1 : (int)ld);
        if constexpr (KC && !PART) {
            x = buffer_load4(rsrc, off);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int soff = 4 * e * (KC ? 1 : (int)ld);
                if constexpr (PART)
                    x[e] = buffer_load1(rsrc, k + dk + e < kend ? off + soff : kOutOfRange);
                else
                    x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, soff, 0));
            }
        }
        if constexpr (ONES) {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = s.one ? (PART && k + dk + e >= kend ? 0.0f : 1.0f) : x[e];
        }
    }

    // The operand from k on. (Kept scalar: the compiler may hold a uniform loop
    // value in vector registers, and would then loop over the lanes of every
    // load.)
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t at_k(int64_t k) const {
        const uint64_t at = (uint64_t)(base + (KC ? k : k * ld));
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
        return buffer_rsrc((const float*)((uint64_t)hi << 32 | lo), 0x80000000ll);
    }

    // Loads unit i of the k-tile at k0. PART: elements at or past kend read
    // zero.
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&r)[2], int i, int64_t k0, int64_t kend,
                                         int tid) const {
        int row, q;
        split_pos<BMN, BK, KC, NT>(i, tid, row, q);
        const auto rsrc = at_k(k0);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int kk = half * (BK / 2);  // k of the unit's half, less 4q
            if constexpr (KC && !PART) {
                r[half] = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[i] + kk * 4, 0, 0));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int soff = (kk + e) * 4 * (KC ? 1 : (int)ld);
                    if constexpr (PART)
                        r[half][e] = buffer_load1(
                            rsrc, k0 + kk + 4 * q + e < kend ? off[i] + soff : kOutOfRange);
                    else
                        r[half][e] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off[i], soff, 0));
                }
            }
        }
    }
};

// The 32 x 32 block at (m0, n0) of the tile over [kbeg, kend) on the f32
// instructions, operands from global memory (the exceptions above: any inputs,
// no staging). A step takes 16 k values, 8 of each operand a lane; the next two
// steps' loads are in flight meanwhile. It is bound by the latency of those
// loads where a few blocks are redone, by the L1 lines they touch where all
// are. Time of a call, us, with ordinary inputs / one row of NaN / NaN
// throughout (the values one by one, a step ahead: in brackets):
//   NN 4096^3              600 / 773 / 1715   (1868, 5857)
//   NT 1000 x 1333 x 777    26 / 47 / 51      (103, 138)
//   TN 2048 x 2048 x 512    28 / 55 / 80      (101, 131)
//   NT 64 x 576 x 100352    66 / 121 / 156    (279, 465)
//   64->128 3x3 32 x 32^2   41 / 92 / 89 and 49 / 117 / 116   (234, 336)
// Inputs that drop bits in one row or throughout cost the same.
template <class OA, class OB>
__device__ __forceinline__ f32x16 f32_block(const OA& oa, const OB& ob, int m0, int n0, int64_t kbeg,
                                            int64_t kend, int lane) {
    const int h = lane >> 5, l32 = lane & 31;
    const auto sa = oa.spot(m0 + l32);
    const auto sb = ob.spot(n0 + l32);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    constexpr int kAhead = 3;  // steps in registers
    f32x4 x[kAhead][2], y[kAhead][2];
    auto load = [&](f32x4(&a)[2], f32x4(&b)[2], int step, auto part) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            oa.template four<decltype(part)::value>(a[u], sa, kbeg + 16 * step, 8 * h + 4 * u, kend);
            ob.template four<decltype(part)::value>(b[u], sb, kbeg + 16 * step, 8 * h + 4 * u, kend);
        }
    };
    auto multiply = [&](const f32x4(&a)[2], const f32x4(&b)[2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][e], b[u][e], acc, 0, 0, 0);
    };
    constexpr std::integral_constant<bool, true> yes{};
    constexpr std::integral_constant<bool, false> no{};
    const int full = (int)((kend - kbeg) / 16);
    if (full > 0) {  // (the last whole step again, unused, past the end)
#pragma unroll
        for (int u = 0; u < kAhead - 1; ++u) load(x[u], y[u], min(u, full - 1), no);
    }
#pragma unroll 1
    for (int t = 0; t < full; t += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            constexpr int d = kAhead - 1;
            load(x[(u + d) % kAhead], y[(u + d) % kAhead], min(t + u + d, full - 1), no);
            if (t + u < full) multiply(x[u], y[u]);  // uniform
        }
    }
    if (kbeg + 16 * (int64_t)full < kend) {
        load(x[0], y[0], full, yes);
        multiply(x[0], y[0]);
    }
    return acc;
}

// The tile at (m0, n0) over [kbeg, kend) of the product of the initialised
// operands oa (rows) and ob (columns), stored by p's epilogue.
template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS, bool TWO, class OA, class OB>
__device__ __forceinline__ void split_tile(const GemmArgs& p, u32x4* smem, OA& oa, OB& ob,
                                           int64_t m0, int64_t n0, int64_t kbeg, int64_t kend,
                                           int slice, int64_t batch) {
    using C_ = SplitCfg<BM, BN, BK, WAVES_M, WAVES_N, KS>;
    constexpr int FM = C_::FM, FN = C_::FN, NT = C_::NT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kset = wave_id / (WAVES_M * WAVES_N);  // k-split wave set
    const int wave = wave_id - kset * (WAVES_M * WAVES_N);
    const int h = lane >> 5, l32 = lane & 31;
    const int wm0 = (wave / WAVES_N) * C_::WM, wn0 = (wave % WAVES_N) * C_::WN;

    f32x16 acc[FM][FN], lo[TWO ? FM : 1][TWO ? FN : 1];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0.0f;
                if constexpr (TWO) lo[i][j][r] = 0.0f;
            }
    f32x4 ra[C_::UA][2], rb[C_::UB][2];

    const int ntiles = (int)((kend - kbeg + BK - 1) / BK);
    // Tile t of the slice goes through the staging registers into LDS buffer
    // t % 2. Units are numbered A's first.
    constexpr bool kMasked = OA::kMasked && OB::kMasked;
    const int nfull = kMasked ? ntiles : (int)((kend - kbeg) / BK);
    constexpr int kUnits = C_::UA + C_::UB;
    // One word for all of a thread's units where they are of one row: with a word
    // each, the registers that the 64x128 convolution tile had left cost it 6%
    // (128 -> 128 channels 3x3, N 21 20^2: 48.1 us, shared 44.8).
    constexpr int kFirstB = !OA::kKC && NT % BM == 0 ? 1 : C_::UA;
    constexpr int kSticky = kFirstB + (!OB::kKC && NT % BN == 0 ? 1 : C_::UB);
    auto word = [](int un) constexpr {
        return un < C_::UA ? (un < kFirstB ? un : kFirstB - 1)
                           : (un - C_::UA < kSticky - kFirstB ? kFirstB + un - C_::UA : kSticky - 1);
    };
    uint32_t sticky[kSticky];
#pragma unroll
    for (int w = 0; w < kSticky; ++w) sticky[w] = 0;
    auto load_unit = [&](int t, int un, auto part) {
        constexpr bool PART = decltype(part)::value;
        const int64_t k0 = kbeg + (int64_t)t * BK;
        if (un == 0) {
            oa.begin(k0, tid);
            ob.begin(k0, tid);
        }
        if (un < C_::UA)
            oa.template load<PART>(ra[un], un, k0, kend, tid);
        else
            ob.template load<PART>(rb[un - C_::UA], un - C_::UA, k0, kend, tid);
    };
    constexpr std::integral_constant<bool, true> yes{};
    constexpr std::integral_constant<bool, false> no{};
    auto load_all = [&](int t) {
        if (t < nfull) {  // uniform
#pragma unroll
            for (int un = 0; un < kUnits; ++un) load_unit(t, un, no);
        } else {
#pragma unroll
            for (int un = 0; un < kUnits; ++un) load_unit(t, un, yes);
        }
    };
    // Step x of splitting a tile: step x % kSplitSteps of unit x / kSplitSteps,
    // the last one of a unit storing its pieces to LDS.
    constexpr int kSteps = kSplitSteps * kUnits;
    SplitState st;
    auto split_step = [&](int t, auto xc) {
        constexpr int x = decltype(xc)::value, un = x / kSplitSteps;
        constexpr bool in_a = un < C_::UA;
        constexpr int i = in_a ? un : un - C_::UA;
        if constexpr (!in_a && OB::kFix && x % kSplitSteps == 0) ob.fix(rb[i], i);
        st.template step<x % kSplitSteps>(in_a ? ra[i] : rb[i], sticky[word(un)],
                                          in_a ? OA::kOnes && ((oa.ones >> i) & 1u)
                                               : OB::kOnes && ((ob.ones >> i) & 1u));
        if constexpr (x % kSplitSteps == kSplitSteps - 1) {
            int row, q;
            if (in_a)
                split_pos<BM, BK, OA::kKC, NT>(i, tid, row, q);
            else
                split_pos<BN, BK, OB::kKC, NT>(i, tid, row, q);
            u32x4* dst = smem + (t & 1) * C_::STAGE + (in_a ? 0 : 3 * C_::PLANE_A);
            const int at = split_unit<BK>(row, q);
#pragma unroll
            for (int p = 0; p < 3; ++p) dst[p * (in_a ? C_::PLANE_A : C_::PLANE_B) + at] = st.piece[p];
        }
    };
    auto split_all = [&](int t) {
        static_for<kSteps>([&](auto xc) { split_step(t, xc); });
    };
    // Tile t reduced from its LDS buffer. With SPLIT, tile t + 1 goes from the
    // registers into the other buffer meanwhile, and each unit's registers
    // then take tile t + 2 (the last whole tile again, unused, past the end:
    // the loop has no branch, so the compiler waits only for the unit it
    // splits). The instruction order is this source's (scheduling barriers):
    // a wave alone on its SIMD overlaps its vector instructions with a matrix
    // instruction only if they follow it closely. The first quarter of the
    // split fills the wait for the operand reads, the rest is spread over the
    // first three quarters of the matrix instructions, so that its LDS stores are
    // done at the barrier; the next row block's operands are read before the
    // current one's products.
    auto reduce = [&](int t, auto split) {
        constexpr bool SPLIT = decltype(split)::value;
        constexpr int S = BK / 16 / KS, NM = 6 * FM * FN * S, ND = SPLIT ? kSteps : 0, HEAD = ND / 4;
        constexpr int NS = NM * 3 / 4;
        const int tl = min(t + 2, nfull - 1);
        auto step = [&](auto xc) {
            constexpr int x = decltype(xc)::value;
            split_step(t + 1, xc);
            if constexpr (x % kSplitSteps == kSplitSteps - 1) load_unit(tl, x / kSplitSteps, no);
        };
        const u32x4* sa = smem + (t & 1) * C_::STAGE;
        const u32x4* sb = sa + 3 * C_::PLANE_A;
        bf16x8 bf[3][FN], af[3];
        auto read_b = [&](int s, int x) {  // piece x of B of step s
#pragma unroll
            for (int j = 0; j < FN; ++j)
                bf[x][j] = __builtin_bit_cast(
                    bf16x8, sb[x * C_::PLANE_B +
                               split_unit<BK>(wn0 + 32 * j + l32, 2 * (kset * S + s) + h)]);
        };
        auto read_a = [&](int g, int x) {  // piece x of group g: step g / FM, row block g % FM
            const int s = g / FM, i = g % FM;
            af[x] = __builtin_bit_cast(
                bf16x8, sa[x * C_::PLANE_A +
                           split_unit<BK>(wm0 + 32 * i + l32, 2 * (kset * S + s) + h)]);
        };
        // The products of a group, ordered so that a piece is read over as its
        // last product is issued (kFreeA, kFreeB) two or more products before
        // the next group or step multiplies it.
        constexpr int kA[6] = {2, 1, 0, 0, 1, 0}, kB[6] = {0, 0, 0, 1, 1, 2};
        constexpr int kFreeA[6] = {2, -1, -1, -1, 1, 0}, kFreeB[6] = {-1, -1, 0, -1, 1, 2};
        read_b(0, 0);
#pragma unroll
        for (int x = 2; x >= 0; --x) read_a(0, x);
        read_b(0, 1);
        read_b(0, 2);
        __builtin_amdgcn_sched_barrier(0);
        static_for<HEAD>(step);
        __builtin_amdgcn_sched_barrier(0);
        static_for<NM>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            constexpr int g = m / (6 * FN), x = m / FN % 6, j = m % FN, s = g / FM;
            f32x16& c = TWO && x != 2 ? lo[TWO ? g % FM : 0][TWO ? j : 0] : acc[g % FM][j];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kA[x]], bf[kB[x]][j], c, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int y0 = HEAD + (m < NS ? m : NS) * (ND - HEAD) / NS,
                          y1 = HEAD + (m + 1 < NS ? m + 1 : NS) * (ND - HEAD) / NS;
            static_for<y1 - y0>([&](auto yc) {
                step(std::integral_constant<int, y0 + decltype(yc)::value>{});
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (j == FN - 1 && g + 1 < S * FM) {
                if constexpr (kFreeA[x] >= 0) read_a(g + 1, kFreeA[x]);
                if constexpr (kFreeB[x] >= 0 && (g + 1) % FM == 0) read_b(s + 1, kFreeB[x]);
            }
        });
    };
    load_all(0);
    split_all(0);
    if (ntiles > 1) load_all(min(1, nfull));
    __syncthreads();
    int t = 0;
    for (; t + 1 < nfull; ++t) {
        reduce(t, yes);
        __syncthreads();
    }
    // the last whole tile and a partial one
    for (;; ++t) {
        const bool last = t + 1 == ntiles;  // uniform
        if (!last && nfull > 0) load_all(nfull);
        reduce(t, no);
        if (last) break;
        split_all(t + 1);
        __syncthreads();
    }

    // The wave sets' halves of the sum meet in LDS: with two column blocks a
    // wave each set finishes one of them, else the first set finishes.
    constexpr bool kShare = KS == 2 && FN % 2 == 0;
    constexpr int FO = kShare ? FN / 2 : FN;  // column blocks the wave finishes
    static_assert(KS == 1 || KS == 2, "wave sets");
    f32x16 out[FM][FO];
    int wo0 = wn0;  // their first column
    if constexpr (TWO) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = acc[i][j] + lo[i][j];
    }
    uint32_t dropped = 0;
#pragma unroll
    for (int w = 0; w < kSticky; ++w) dropped |= sticky[w];
    const bool lost = __syncthreads_or((int)(dropped & 0xffffu));
    // (the barrier above: every wave is done with the staging buffers)
    // A bit for each row and column of the tile with dropped bits, past what
    // the wave sets exchange.
    constexpr int kFlags = (BM + BN) / 32;
    uint32_t* const flags = reinterpret_cast<uint32_t*>(smem + 2 * C_::STAGE) - kFlags;
    if (lost) {  // uniform
        if (tid < kFlags) flags[tid] = 0;
        __syncthreads();
#pragma unroll
        for (int un = 0; un < kUnits; ++un) {
            int row, q;
            if (un < C_::UA)
                split_pos<BM, BK, OA::kKC, NT>(un, tid, row, q);
            else
                split_pos<BN, BK, OB::kKC, NT>(un - C_::UA, tid, row, q);
            if (un >= C_::UA) row += BM;
            if (sticky[word(un)] & 0xffffu) atomicOr(flags + row / 32, 1u << (row % 32));
        }
        __syncthreads();
    }
    if constexpr (KS == 1) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) out[i][j] = acc[i][j];
    } else {
        float* x = reinterpret_cast<float*>(smem);
        constexpr int WS = WAVES_M * WAVES_N, BLK = FM * FO * 1024;
        static_assert((kShare ? 2 : 1) * WS * BLK * 4 + kFlags * 4 <= 2 * C_::STAGE * 16,
                      "k-split LDS space");
        if (kShare || kset == 1) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FO; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        x[(kShare ? kset * WS + wave : wave) * BLK + (i * FO + j) * 1024 + r * 64 + lane] =
                            kShare ? (kset ? acc[i][j][r] : acc[i][j + FO < FN ? j + FO : 0][r])
                                   : acc[i][j][r];
        }
        __syncthreads();
        if (!kShare && kset == 1) return;  // uniform; no barrier follows
        const int from = kShare ? (1 - kset) * WS + wave : wave;
        wo0 = wn0 + (kShare ? 32 * FO * kset : 0);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FO; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float own =
                        kShare && kset ? acc[i][j + FO < FN ? j + FO : 0][r] : acc[i][j][r];
                    const float other = x[from * BLK + (i * FO + j) * 1024 + r * 64 + lane];
                    // set 0's half first, as the sum does not depend on the finisher
                    out[i][j][r] = kset ? other + own : own + other;
                }
    }

    // The exceptions: rows and columns with dropped bits, and results that are
    // not finite (bit i * FO + j of `redo`: the block has any).
    uint32_t redo = 0;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FO; ++j) {
            float finite = 0.0f;  // 0 while every result is finite, else NaN
#pragma unroll
            for (int r = 0; r < 16; ++r) finite = fmaf(out[i][j][r], 0.0f, finite);
            if (__any(finite != 0.0f) ||
                (lost && (flags[wm0 / 32 + i] | flags[(BM + wo0) / 32 + j])))
                redo |= 1u << (i * FO + j);
        }
    redo = __builtin_amdgcn_readfirstlane(redo);
    // (expected not to be taken: else its scalars are spilled around the k loop)
    while (__builtin_expect(redo != 0, 0)) {  // uniform
        const int b = __builtin_ctz(redo), bi = b / FO, bj = b % FO;
        redo &= redo - 1;
        const f32x16 f = f32_block(oa, ob, wm0 + 32 * bi, wo0 + 32 * bj, kbeg, kend, lane);
        uint32_t rows = lost ? flags[wm0 / 32 + bi] : 0;
        if (lost && ((flags[(BM + wo0) / 32 + bj] >> l32) & 1u)) rows = ~0u;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FO; ++j)
                if (b == i * FO + j) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (((rows >> (8 * (r / 4) + 4 * h + r % 4)) & 1u) ||
                            !(fabsf(out[i][j][r]) <= FLT_MAX))
                            out[i][j][r] = f[r];
                }
    }

    const TileOut<FO> to = tile_out<BM, BN, FO>(p, m0, n0, wm0, wo0, h, l32, slice, batch);
    const float none[1][1][16] = {};
    tile_store<FM, FO, false>(p, to, out, none, n0 + wo0 + l32);
}

// split_tile of a dense problem.
template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS, bool TWO, bool AK, bool BKC>
__device__ __forceinline__ void split_dense(const GemmArgs& p, u32x4* smem, int64_t m0, int64_t n0,
                                            int64_t kbeg, int64_t kend, int slice, int64_t batch) {
    using C_ = SplitCfg<BM, BN, BK, WAVES_M, WAVES_N, KS>;
    SplitOperand<BM, BK, AK, C_::NT, C_::UA, !AK> oa;
    SplitOperand<BN, BK, BKC, C_::NT, C_::UB> ob;
    oa.init(p.A + batch * p.sA, p.lda, m0, p.M, p.sum_row ? p.M : -1, threadIdx.x);
    ob.init(p.B + batch * p.sB, p.ldb, n0, p.N, -1, threadIdx.x);
    split_tile<BM, BN, BK, WAVES_M, WAVES_N, KS, TWO>(p, smem, oa, ob, m0, n0, kbeg, kend, slice,
                                                      batch);
}

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int KS, bool TWO, bool AK, bool BKC>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N * KS, 2) void gemm_split_kernel(GemmArgs p) {
    using C_ = SplitCfg<BM, BN, BK, WAVES_M, WAVES_N, KS>;
    __shared__ u32x4 smem[2 * C_::STAGE];
    int bid = blockIdx.x, slice = blockIdx.y;
    if (gridDim.y > 1 && (gridDim.x & 7) != 0)
        split_coords(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x, gridDim.y, bid, slice);
    int tm, tn;
    tile_coords(p, bid, tm, tn);
    const int64_t kbeg = (int64_t)slice * p.k_per_slice;
    split_dense<BM, BN, BK, WAVES_M, WAVES_N, KS, TWO, AK, BKC>(p, smem, (int64_t)tm * BM, (int64_t)tn * BN,
                                                      kbeg, min(p.K, kbeg + p.k_per_slice), slice,
                                                      blockIdx.z);
}

// Several independent dense GEMMs in one launch (the products of one
// backward step, or projections of one input): problem q owns workgroups
// [first[q], first[q] + tiles_q * slices[q]) of a 1-D grid, each range
// starting at a multiple of 8 so that a workgroup's XCD is its id within the
// problem modulo 8, as in a launch of its own (ids past a problem's range,
// the padding up to the next multiple of 8, exit at once). The problems'
// workgroups share the CUs (three fit), so one problem's load latency,
// barriers and epilogue overlap another's products; one launch per GEMM
// leaves each CU a single workgroup of small tiles whose waves all stall at
// the same points.
template <int BM, int BN, int BK, int WAVES_M, int WAVES_N>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 3) void gemm_split_group_kernel(GemmGroupArgs g) {
    using C_ = SplitCfg<BM, BN, BK, WAVES_M, WAVES_N, 1>;
    __shared__ u32x4 smem[2 * C_::STAGE];
    const int b = blockIdx.x;
    int q = 0;
#pragma unroll
    for (int i = 1; i < kGroupMax; ++i)
        if (i < g.count && b >= g.first[i]) q = i;
    const GemmArgs& p = g.prob[q];
    const int tiles = p.tiles_m * p.tiles_n, slices = g.slices[q];
    const int lin = b - g.first[q];
    if (lin >= tiles * slices) return;  // uniform: padding up to the next problem
    int bid, slice, tm, tn;
    split_coords(lin, tiles, slices, bid, slice);
    tile_coords(p, bid, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int64_t kbeg = (int64_t)slice * p.k_per_slice, kend = min(p.K, kbeg + p.k_per_slice);
    switch (g.layout[q]) {
        case NRS_NN:
            split_dense<BM, BN, BK, WAVES_M, WAVES_N, 1, true, true, false>(p, smem, m0, n0, kbeg,
                                                                           kend, slice, 0);
            break;
        case NRS_NT:
            split_dense<BM, BN, BK, WAVES_M, WAVES_N, 1, true, true, true>(p, smem, m0, n0, kbeg,
                                                                          kend, slice, 0);
            break;
        default:
            split_dense<BM, BN, BK, WAVES_M, WAVES_N, 1, true, false, false>(p, smem, m0, n0, kbeg,
                                                                            kend, slice, 0);
            break;
    }
}

}  // namespace nrs
