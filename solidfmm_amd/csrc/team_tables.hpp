// Swap blocks in matrix-core operand order for the team kernels (team.hpp).
//
// The folded blocks of degree n couple orders of one parity only: the real
// part of an output order m takes inputs l = m + n (mod 2), the imaginary
// part l = m + n + 1 (operator_data.cpp:47-147).  Split by the parity of the
// input order (class e: l = 2i + e), each degree is four dense blocks of
// about half its size, numbered 2 part + e; the output class of the real
// blocks is e + n, of the imaginary ones e + n + 1 (mod 2).
//
// With NJ = n/8 + 1 chunks of four indices per class, a block is cut into
//   NJ <= kSmall  NJ x NJ operands of v_mfma_f64_4x4x4_4b_f64, 16 doubles
//                 each: entry i + 4 k of operand (o, c) is output index
//                 4 o + i, input index 4 c + k.  Operands are stored two by
//                 two, entry by entry, so a lane reads a pair at once;
//   NJ > kSmall   operands of v_mfma_f64_16x16x4_f64, 64 doubles each: entry
//                 r + 16 k of operand (b, c) is output index 16 b + r, input
//                 index 4 c + k.
// Entries outside a block are zero.
//
// Two tables follow each other: the blocks as they stand (M-type pipelines)
// and their transposes D^-1 S^T D, D = diag(1, 2, ..., 2) (L-type).
#pragma once

#include <cstddef>

#include "mfma_tables.hpp"

namespace sfmm {
namespace team {

constexpr int chunks(int n) { return n / 8 + 1; }
// The two instructions cost the same per product (16 and 64 clocks); the
// small one wastes nothing on classes of fewer than 16 orders.
inline constexpr int kSmall = 3;
constexpr int row_blocks(int nj) { return (nj + 3) / 4; }
// doubles of one degree with nj chunks
constexpr int degree_size(int nj) { return nj <= kSmall ? 64 * nj * nj : 256 * row_blocks(nj) * nj; }
// first double of the degrees with nj chunks (8 degrees share a chunk count)
constexpr int base_of(int nj)
{
    int s = 0;
    for (int j = 1; j < nj; ++j) s += 8 * degree_size(j);
    return s;
}
// orders the team kernels take
inline constexpr int kMaxOrder = 48;
constexpr int table_size() { return base_of(chunks(kMaxOrder - 1) + 1); }

// Both tables (2 table_size() doubles) on the current device, built on first
// use and kept until the process ends; nullptr on failure (swap_host.cpp).
const double *device_table();

}  // namespace team
}  // namespace sfmm
