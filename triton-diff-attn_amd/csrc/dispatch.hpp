// The launch geometry of a forward as a pure function of its sizes and options.  Plain C++: a test compiles it by itself.
#pragma once

namespace da_abi {

constexpr int kNumCU = 256;

// Whether a forward runs in 64-row, four-wave workgroups instead of 128-row ones.  (The reference autotunes its tiles per
// (N, D, Dv), src/kernel.py:12-19; there is no tuning state here.)  `n`: the padded sequence length, a multiple of 128;
// `blocks`: B*H*n/128.  Figures: us of a launch, 128-row -> 64-row.
// Blocks of one length: up to 128 of them, i.e. where 128-row blocks leave half of the chip idle (bf16, D <= 64, B1 H8
// N2000 D64 39.6 -> 33.8, with dropout 57.7 -> 41.1; D32 29.3 -> 23.3).  The rings of a D >= 64 workgroup fill a CU's LDS
// whatever its rows, so from 129 on the halves take a second round (bf16, B1 H9 N2048 D64 38.3 -> 56.8, B1 H12 N2048 D64
// 41.4 -> 56.9, D128 75 -> 105).
// Causal blocks differ in length and end with the longest; halves, longest first, are shorter and dealt more evenly.
//   D32, two workgroups to a CU: up to 256 (bf16, B1 H8 N2048 29.0 -> 22.4, B1 H16 N2048 29.4 -> 25.3; fp16, 256 blocks of
//   N = 256 9.2 -> 8.0, N = 128 7.4 -> 7.6).
//   D64 and D128: the second round, of the shortest halves, has to fit beside the first.  A unit of one or two blocks
//   has no short ones, and a workgroup's start and end, which do not shrink with N, are most of it; the longer the unit, the
//   further up the halves win.  The blocks at which the two meet, measured in fp16: D64 130 at N <= 256, 145 at 512, 150 at 768,
//   190 at 1024, 235 at 1536, above 256 at 2048 (192 blocks: N = 128 9.7 -> 15.2, 256 12.5 -> 17.3, 512 16.4 -> 19.6, 1024
//   24.0 -> 24.4, 2048 39.4 -> 33.9); D128 130 at N <= 256, 165 at 512 and 640, 200 at 768, 215 at 1024, 255 at 1536 (192
//   blocks: N = 128 16.4 -> 21.6, 512 26.8 -> 28.7, 1024 40.5 -> 37.9, 2048 68.8 -> 59.1).  The two lines below lie on or
//   just under them.  Beyond: bf16, B1 H4 N8192 D64 139 -> 116, 384 blocks D64 46 -> 61, B1 H32 N3001 D128 230 -> 328.
constexpr bool fwd_64_rows(int d, bool causal, int n, long long blocks) {
  int limit = kNumCU / 2;
  if (causal && d == 32) limit = kNumCU;
  if (causal && d == 64 && n > 512) limit += (n - 512) / 12;
  if (causal && d == 128 && n > 256) limit += (n - 256) / 8;
  const int most = d == 128 ? kNumCU - 1 : kNumCU;
  return blocks <= (limit < most ? limit : most);
}

}  // namespace da_abi
