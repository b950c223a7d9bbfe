// What the rules of the kernels that cut K over a workgroup's waves share (qmm_gemm_w4k.hip,
// qmm_gemm_w4a8k.hip, qmm_gemm_b8k.hip, qmm_gemm_f16w8k.hip): host work only.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace qmm {

// The row blocks of a column block run one after another on an XCD, and every column block
// reads all rows again: with many long rows these no longer come from an L2, and a round of
// workgroups takes longer than its K says. The factor: 1 up to 8 million values, 1 + by from 16
// million on (f16, 64 x 64 results, priced without / measured: 1473 x 14464 x 1344 90 / 124 us,
// 2102 x 9216 x 816 60 / 81).
inline double many_rows(int M, int K, double by) {
    const double values = (double)M * K / (8 << 20);
    return 1 + by * std::min(1.0, std::max(0.0, std::log2(values)));
}

} // namespace qmm
