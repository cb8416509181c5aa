"""Host build of what the e4m3 down pass works out of a group's number (csrc/block_groups.h): the block it belongs to
and where its weight rows and scales lie."""
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


def _run(tmp_path, source):
    (tmp_path / "main.cpp").write_text(source)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, "main.cpp", "-o", "main"], cwd=tmp_path)
    return subprocess.run([str(tmp_path / "main")], check=True, capture_output=True, text=True, timeout=120).stdout


def test_every_group_has_its_block(tmp_path):
    assert _run(tmp_path, _BLOCKS) == ""


def test_rows_of_a_block_without_an_expert_are_inside_the_tensor(tmp_path):
    assert _run(tmp_path, _ROWS) == ""
