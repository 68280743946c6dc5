"""The workgroup order of the multi-pass convolution's fused column and row pass (csrc/longmap.hpp),
checked by a host program built from the same header: every pair and group of rows exactly once, and the
workgroups that read the same input on one XCD (consecutive workgroups go to the 8 XCDs in turn)."""
import shutil
import subprocess

import pytest

import sffft_amd as sf

PROGRAM = r"""
#include <cstdio>
#include <set>
#include <utility>
#include <vector>

#include "longmap.hpp"

using namespace sffft;

// pairs whose workgroups are not all on one XCD
template <int GROUPS>
int split_pairs(int nch, int BP, bool grouped) {
  const int n = nch * BP * GROUPS;
  std::vector<int> seen(n, 0);
  std::vector<std::set<int>> xcds(nch * BP);
  for (int i = 0; i < n; i++) {
    const FusedBlock b = fused_block<GROUPS>(i, nch, BP, grouped);
    if (b.c < 0 || b.c >= nch || b.bp < 0 || b.bp >= BP || b.kt < 0 || b.kt >= GROUPS) return -1;
    if (seen[(b.c * BP + b.bp) * GROUPS + b.kt]++) return -1;
    xcds[b.c * BP + b.bp].insert(i & 7);
  }
  int split = 0;
  for (const auto& x : xcds) split += x.size() > 1;
  return split;
}

template <int GROUPS>
bool check() {
  for (int nch = 1; nch < 90; nch++)
    for (int BP = 1; BP < 40; BP += BP < 9 ? 1 : 6) {
      if (split_pairs<GROUPS>(nch, BP, false) < 0) return printf("in order: GROUPS=%d nch=%d BP=%d\n", GROUPS, nch, BP), false;
      const int split = split_pairs<GROUPS>(nch, BP, true);
      if (split < 0 || split >= 8) return printf("grouped: GROUPS=%d nch=%d BP=%d: %d\n", GROUPS, nch, BP, split), false;
      if (nch % 8 == 0 && split) return printf("GROUPS=%d nch=%d BP=%d: %d\n", GROUPS, nch, BP, split), false;
      if (nch * BP * GROUPS > 256 && !fused_grouped(nch * BP * GROUPS, nch)) return printf("not grouped\n"), false;
    }
  return true;
}

int main() {
  if (!check<1>() || !check<2>() || !check<4>()) return 1;
  // the launches: half a round of workgroups at least, and no second round of few but for 64x32x32
  const bool ok = !fused_launch(127, 64, 32) && fused_launch(128, 64, 32) && fused_launch(257, 64, 32) &&
                  !fused_launch(127, 64, 64) && fused_launch(256, 64, 64) && !fused_launch(257, 64, 64) &&
                  !fused_launch(303, 64, 64) && fused_launch(304, 64, 64) && !fused_launch(303, 16, 32) &&
                  fused_launch(304, 16, 32) && !fused_launch(1ll << 31, 64, 32);
  return ok ? 0 : 2;
}
"""


def test_workgroup_order(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    src = tmp_path / "order.cpp"
    src.write_text(PROGRAM)
    csrc = sf.LIB_PATH.rsplit("/", 1)[0] + "/csrc"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", csrc, "-o", str(tmp_path / "order"), str(src)], check=True)
    r = subprocess.run([str(tmp_path / "order")], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout)
