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

// A share of the groups, [begin, end), none of them empty.  One of a block and more is walked from the first block that starts
// in it, and its groups in front of that block come last: workgroups whose blocks are one expert's then read the same weight
// rows at about the same time, wherever their shares were cut.  (Shares shorter than a block don't all hold a block's start.)
// Places of the walk are 0 .. count - 1.
struct BlockShare {
  int begin, count, lead, per_block, lead_block, end_block;   // `lead` groups, all of lead_block, come last

  static constexpr BlockShare of(int begin, int end, int per_block, uint32_t rcp) {
    const int mb = block_of_group(begin, per_block, rcp), behind = (mb + 1) * per_block - begin;
    const bool turned = behind < per_block && end - begin >= per_block;
    return {begin, end - begin, turned ? behind : 0, per_block, mb, block_of_group(end - 1, per_block, rcp)};
  }
  // The group at a place.
  constexpr int group(int place) const { return begin + place + (place < count - lead ? lead : lead - count); }
  constexpr int first_block() const { return lead ? lead_block + 1 : lead_block; }
  constexpr bool last(int mb) const { return mb == (lead ? lead_block : end_block); }
  // The block behind one that is not the last.
  constexpr int next(int mb) const { return mb == end_block ? lead_block : mb + 1; }
  // The first place behind a block's, and how far the places of a block's groups lie in front of their numbers in it.
  constexpr int stop(int mb) const {
    return last(mb) ? count : mb == end_block ? count - lead : (mb + 1) * per_block - begin - lead;
  }
  constexpr int shift(int mb) const { return begin + lead - (lead && mb == lead_block ? count : 0) - mb * per_block; }
};
