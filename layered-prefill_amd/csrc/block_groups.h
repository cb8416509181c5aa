// Where a group of weight rows of a pass over (block, sixteen rows) groups lies.  Plain functions of numbers (constexpr, so for
// host and device alike): what the launch works out and what the kernel makes of it.
#pragma once

#include <cstdint>

// 2^32 / groups per block, rounded up.  That of one group per block has no place in 32 bits: block_of_group does not look at it.
constexpr uint32_t block_groups_rcp(int per_block) {
  return per_block == 1 ? 0 : static_cast<uint32_t>((1LL << 32) / per_block + 1);
}

// g / per_block for group numbers below 2^30.
constexpr int block_of_group(int g, int per_block, uint32_t rcp) {
  if (per_block == 1) return g;
  const int mb = static_cast<int>(static_cast<uint64_t>(static_cast<uint32_t>(g)) * rcp >> 32);  // the quotient, or one more
  return mb * per_block > g ? mb - 1 : mb;
}

// Elements from expert 0's first row to row `row` of expert e.  A block that a caller's alignment gives to no expert (-1) holds
// no slots; what is read on its account and never used comes out of expert 0.
constexpr int64_t expert_row(int e, int row, int64_t stride_e, int64_t stride_row) {
  return (e < 0 ? 0 : e) * stride_e + row * stride_row;
}
