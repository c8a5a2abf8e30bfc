// Answers what the planner of the split GEMM (gemm_plan.hpp) decides, one line
// of output per line of input. The layouts are NN, NT, TN; sizes are integers.
//   gemm LAYOUT M N K BATCH ROW_OF_SUMS SPLIT_K CUS  ->  "BMxBNxBK SLICES K_PER_SLICE" or "f32"
//     (of operands 16-byte aligned)
//   group LAYOUT M N K ROW_OF_SUMS                   ->  1 if the group kernel takes it
//   shared ROWS INNER COLS                           ->  1 if the shared-lhs backward runs as a group
#include <iostream>
#include <sstream>
#include <string>

#include "gemm_plan.hpp"

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
