// What a product that leaves its norm half done (gemm_strips.hip) and the product that reads its rows (gemm_rows.hip) agree on: up
// to kScaledRows rows, and kRowSums places a row in memory for its sums of squares, of which the first so many are written.
#pragma once

namespace arle {

constexpr int kScaledRows = 8;
constexpr int kRowSums = 256;

}  // namespace arle
