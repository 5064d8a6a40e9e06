// The columns that a thread of gemm_f32_split.hip loads, for the kernel and for a check of their range on the host.
#pragma once

namespace oamd {

// First of the eight columns that thread `lc` of a row's four loads of the 32-column piece at column k of K (a multiple of 16). Past the
// row's end the row's first columns, which are cleared or never used: no load leaves its row.
constexpr int split_column(int k, int lc, int K) { return k + 8 * lc < K ? k + 8 * lc : 0; }

}  // namespace oamd
