// Which launches of the multi-pass convolution run the column and row passes in one kernel
// (long_cols_rows), and which pair and rows a workgroup of that kernel takes. Plain C++ (constexpr
// functions, for host and device), so that a host program can check it.
#pragma once

namespace sffft {

// Launches of at least 128 workgroups, half the CUs: one workgroup takes some 20 us however few they are,
// where the separate passes spread their columns and rows over all CUs. L=65536 bf16, separate -> fused:
// B=2 H=16 (64 workgroups) 28.1 -> 28.8 us, H=32 (128) 33.6 -> 31.1, H=64 51.6 -> 39.7; L=32768 H=32 (128)
// 25.5 -> 19.8. A second round of few workgroups takes as long as a full one: from 257 to some 300 the
// separate passes are 1 to 5% faster (separate against fused, 64x64x32 at 260 workgroups 55.5 against 57.5 us,
// 280 56.2 / 57.4, 308 60.4 / 58.9; 16x64x32 at 260 48.9 / 51.5; 16x32x32 at 280 29.0 / 30.1), but for
// 64x32x32 (34.8 / 33.3).
constexpr int LF_MIN_BLOCKS = 128, LF_ROUND = 256, LF_SECOND = 304;
constexpr bool fused_launch(long long blocks, int nc, int r0) {
  if (blocks < LF_MIN_BLOCKS || blocks > 0x7fffffff) return false;
  return blocks <= LF_ROUND || blocks >= LF_SECOND || (nc == 64 && r0 == 32);
}

// Workgroup i -> channel slot c of the chunk's nch, pair bp of its BP, group kt of 16 rows. Consecutive
// workgroups go to the 8 XCDs in turn. Grouped, the GROUPS workgroups of a pair, which read the same
// input, and the pairs of a channel, which read the same spectrum, follow each other on one XCD: whole
// channels in turn over the XCDs; of the channels that remain an eighth of their pairs each; the last, fewer
// than 8, pairs in order. In order otherwise: pairs and channels over all XCDs.
//
// Chunks of 8 n channels are grouped as ever. Others from the second round on, when the bytes count: in
// order -> grouped, bf16, L=65536 B=64 H=4 90.3 -> 68.8 us, B=10 H=300 914 -> 868, L=32768 B=2 H=301 103 -> 95.6,
// B=10 H=301 463 -> 429. With fewer workgroups than CUs their loads are not what bounds them, and
// grouped ones ask one L2 for the same lines at once (L=32768 B=10 H=9 20.8 -> 22.5).
struct FusedBlock {
  int c, bp, kt;
};
constexpr bool fused_grouped(int blocks, int nch) { return (nch & 7) == 0 || blocks > LF_ROUND; }
template <int GROUPS>
constexpr FusedBlock fused_block(int i, int nch, int BP, bool grouped) {
  const int per = BP * GROUPS;
  if (!grouped) {
    const int c = i / per, rest = i - c * per, bp = rest / GROUPS;
    return {c, bp, rest - bp * GROUPS};
  }
  const int head = nch & ~7, m = i - head * per;
  if (m < 0) {
    const int j = i >> 3, q = j / per, rest = j - q * per, bp = rest / GROUPS;
    return {8 * q + (i & 7), bp, rest - bp * GROUPS};
  }
  const int each = (nch & 7) * BP >> 3;  // pairs of the rest on each XCD
  const bool dealt = m < 8 * each * GROUPS;
  const int j = dealt ? m >> 3 : m - 8 * each * GROUPS;
  const int pair = (dealt ? (m & 7) * each : 8 * each) + j / GROUPS, c = pair / BP;
  return {head + c, pair - c * BP, j % GROUPS};
}

}  // namespace sffft
