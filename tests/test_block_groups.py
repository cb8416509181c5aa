"""Host build of what the e4m3 down pass works out of a group's number (csrc/block_groups.h): the block it belongs to,
where its weight rows and scales lie, and in which order a share of groups is walked."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "layered-prefill_amd", "csrc")

# Prints the first wrong block of every number of groups per block, or nothing.
_BLOCKS = r"""
#include <cstdio>
#include "block_groups.h"
int main() {
  const int last = (1 << 30) - 1;
  for (int per = 1; per <= 8192; ++per) {
    const uint32_t rcp = block_groups_rcp(per);
    auto wrong = [&](int64_t g) {
      if (g < 0 || g > last || block_of_group(static_cast<int>(g), per, rcp) == g / per) return false;
      std::printf("groups per block %d, group %lld: block %d\n", per, static_cast<long long>(g), block_of_group(static_cast<int>(g), per, rcp));
      return true;
    };
    bool bad = false;
    for (int64_t b = 0, step = 1; b * per <= last && !bad; b += step) {   // both ends of blocks, wider apart as they get more
      bad = wrong(b * per) || wrong(b * per + per - 1);
      if (b >= 512 * step) step *= 2;
    }
    if (!bad) wrong(last);
  }
}
"""

# Prints the rows that lie in front of the tensor or elsewhere than their expert's.
_ROWS = r"""
#include <cstdio>
#include "block_groups.h"
int main() {
  const int64_t strides[][2] = {{2048 * 768, 768}, {2048, 1}, {16LL * (1 << 28), 1 << 28}};
  for (const auto& s : strides)
    for (int e = -1; e < 4; ++e)
      for (int row = 0; row < 16; row += 15) {
        const int64_t want = (e == -1 ? 0 : e * s[0]) + row * s[1], got = expert_row(e, row, s[0], s[1]);
        if (got != want) std::printf("expert %d row %d: %lld\n", e, row, static_cast<long long>(got));
      }
}
"""

# Prints the shares that are not walked as they should be: every group once, block by block in the order that the kernel
# changes blocks, and from a block's first row on where the share is a block long.
_WALKS = r"""
#include <cstdio>
#include <vector>
#include "block_groups.h"
int main() {
  for (int per : {1, 2, 3, 6, 10, 64, 128, 180, 256})
    for (int blocks : {1, 2, 5, 37, 128, 370, 1120, 2168}) {
      const uint32_t rcp = block_groups_rcp(per);
      const int64_t groups = static_cast<int64_t>(blocks) * per;
      std::vector<int> seen(groups, 0);
      for (int share = 0; share < 256; ++share) {
        const int begin = groups * share / 256, end = groups * (share + 1) / 256;
        if (begin >= end) continue;
        const BlockShare walk = BlockShare::of(begin, end, per, rcp);
        bool bad = end - begin >= per && walk.group(0) % per;
        int place = 0, mb = walk.first_block(), turns = 0;
        for (;; mb = walk.next(mb)) {
          for (; place < walk.stop(mb) && !bad; ++place) {
            const int g = walk.group(place);
            if (g < begin || g >= end || g / per != mb || g - mb * per != place + walk.shift(mb) || seen[g]++) bad = true;
            else if (place && g != walk.group(place - 1) + 1 && g != begin) bad = true;
          }
          if (bad || walk.last(mb) || ++turns > blocks) break;
        }
        if (bad || place != end - begin) std::printf("groups per block %d, blocks %d, share %d: place %d of block %d\n", per, blocks, share, place, mb);
      }
      for (int64_t g = 0; g < groups; ++g)
        if (seen[g] != 1) std::printf("groups per block %d, blocks %d: group %lld walked %d times\n", per, blocks, static_cast<long long>(g), seen[g]);
    }
}
"""


def _run(tmp_path, source):
    (tmp_path / "main.cpp").write_text(source)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, "main.cpp", "-o", "main"], cwd=tmp_path)
    return subprocess.run([str(tmp_path / "main")], check=True, capture_output=True, text=True, timeout=120).stdout


def test_every_group_has_its_block(tmp_path):
    assert _run(tmp_path, _BLOCKS) == ""


def test_rows_of_a_block_without_an_expert_are_inside_the_tensor(tmp_path):
    assert _run(tmp_path, _ROWS) == ""


def test_shares_are_walked_from_a_blocks_first_row(tmp_path):
    assert _run(tmp_path, _WALKS) == ""
