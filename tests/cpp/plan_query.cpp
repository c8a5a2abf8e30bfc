// Answers what the planners of the split GEMM (gemm_plan.hpp) and of the
// convolutions (conv_plan.hpp) decide, one line of output per line of input. The
// layouts are NN, NT, TN; sizes are integers.
//   gemm LAYOUT M N K BATCH ROW_OF_SUMS SPLIT_K CUS  ->  "BMxBNxBK SLICES K_PER_SLICE" or "f32"
//     (of operands 16-byte aligned)
//   conv N C_IN C_OUT H W KH KW STRIDE PAD CUS  ->  for the forward and, of stride 1, the input
//     gradient: "BMxBNxBK" if the split tiles are chosen ahead of the others, else "-"
//   group LAYOUT M N K ROW_OF_SUMS                   ->  1 if the group kernel takes it
//   shared ROWS INNER COLS                           ->  1 if the shared-lhs backward runs as a group
#include <iostream>
#include <sstream>
#include <string>

#include "conv_plan.hpp"

static int layout_of(const std::string& s) { return s == "NN" ? NRS_NN : s == "NT" ? NRS_NT : NRS_TN; }

int main() {
    for (std::string line; std::getline(std::cin, line);) {
        std::istringstream in(line);
        std::string what, layout;
        in >> what;
        if (what == "gemm") {
            int64_t m, n, k, batch;
            int sums, split, cus;
            in >> layout >> m >> n >> k >> batch >> sums >> split >> cus;
            nrs::GemmSize s{layout_of(layout), m, n, k, batch, sums != 0, split != 0};
            s.wide = s.lda() % 4 == 0 && s.ldb() % 4 == 0 && (batch == 1 || (m * k % 4 == 0 && n * k % 4 == 0));
            if (!nrs::split_takes(s, cus)) {
                std::cout << "f32\n";
            } else {
                const nrs::SplitPlan p = nrs::plan_split(s, cus);
                const nrs::SplitShape& t = nrs::kSplitShapes[p.tile];
                std::cout << t.bm << "x" << t.bn << "x" << t.bk << " " << p.slices << " "
                          << p.k_per_slice << "\n";
            }
        } else if (what == "conv") {
            nrs::SlabConv f;
            int pad, cus;
            in >> f.N >> f.C >> f.M >> f.H >> f.W >> f.kh >> f.kw >> f.stride >> pad >> cus;
            f.pad_h = f.pad_w = pad;
            f.OH = (f.H + 2 * pad - f.kh) / f.stride + 1;
            f.OW = (f.W + 2 * pad - f.kw) / f.stride + 1;
            nrs::SlabConv d = f;  // the flipped convolution of the output gradient
            std::swap(d.C, d.M);
            std::swap(d.H, d.OH);
            std::swap(d.W, d.OW);
            d.pad_h = f.kh - 1 - pad;
            d.pad_w = f.kw - 1 - pad;
            for (const nrs::SlabConv* s : {&f, &d}) {
                const bool split = nrs::split_conv_better(*s, cus) && nrs::split_conv_takes(*s);
                const nrs::SplitShape& t = nrs::kSplitShapes[nrs::split_conv_tile(*s, cus)];
                if (split && (s == &f || f.stride == 1))
                    std::cout << t.bm << "x" << t.bn << "x" << t.bk;
                else
                    std::cout << "-";
                std::cout << (s == &f ? " " : "\n");
            }
        } else if (what == "group") {
            int64_t m, n, k;
            int sums;
            in >> layout >> m >> n >> k >> sums;
            std::cout << nrs::group_takes(nrs::GemmSize{layout_of(layout), m, n, k, 1, sums != 0}) << "\n";
        } else if (what == "shared") {
            int64_t rows, inner, cols;
            in >> rows >> inner >> cols;
            std::cout << nrs::shared_lhs_fits(rows, inner, cols) << "\n";
        } else {
            std::cout << "unknown query\n";
        }
        if (!in) return 1;
    }
    return 0;
}
