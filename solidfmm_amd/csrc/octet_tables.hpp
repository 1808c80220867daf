// Swap blocks in matrix-core operand order for the octet kernels (octet.hpp).
//
// A degree's folded blocks fall into four dense ones by part and parity of
// the input order, see team_tables.hpp.  One v_mfma_f64_4x4x4_4b_f64 takes
// the real block of class e for its translation blocks 0 and 1 and the
// imaginary block of class e for 2 and 3, so operand (e, o, c) has 32
// doubles: entry i + 4 part + 8 k is output index 4 o + i and input index
// 4 c + k of that part.  With NJ = n/8 + 1 chunks per class, the NJ x NJ
// operands of a class are stored two by two, entry by entry (one by one at
// NJ = 1), padded to an even count.
//
// Two tables follow each other as in team_tables.hpp: M-type, then L-type.
#pragma once

#include "team_tables.hpp"

namespace sfmm {
namespace octet {

using team::chunks;
inline constexpr int kMaxOrder = 24;

// doubles of one class of a degree with nj chunks
constexpr int class_size(int nj) { return nj == 1 ? 32 : 32 * ((nj * nj + 1) & ~1); }
// first double of degree n
constexpr int degree_base(int n)
{
    int s = 0;
    for (int j = 0; j < n; ++j) s += 2 * class_size(chunks(j));
    return s;
}
constexpr int table_size(int orders) { return degree_base(orders); }
// entry i + 4 part + 8 k of operand (e, o, c)
constexpr int entry(int n, int part, int e, int o, int c, int i, int k)
{
    const int nj = chunks(n), at = degree_base(n) + e * class_size(nj), lane = i + 4 * part + 8 * k;
    if (nj == 1) return at + lane;
    const int p = o * nj + c;
    return at + (p / 2) * 64 + lane * 2 + p % 2;
}

// Both tables (2 table_size(kMaxOrder) doubles) on the current device, built
// on first use and kept until the process ends; nullptr on failure.
const double *device_table();

}  // namespace octet
}  // namespace sfmm
