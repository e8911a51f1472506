// The launch geometries of a forward and of a backward as pure functions of the sizes and options.  Plain C++: a test
// compiles it by itself.
#pragma once

namespace da_abi {

constexpr int kNumCU = 256;

// Whether a forward runs in 64-row, four-wave workgroups instead of 128-row ones.  (The reference autotunes its tiles per
// (N, D, Dv), src/kernel.py:12-19; there is no tuning state here.)  `n`: the padded sequence length, a multiple of 128;
// `blocks`: B*H*n/128.  Figures: us of a launch, 128-row -> 64-row.
// Blocks of one length: up to 128 of them, i.e. where 128-row blocks leave half of the chip idle (bf16, D <= 64, B1 H8
// N2000 D64 39.6 -> 33.8, with dropout 57.7 -> 41.1; D32 29.3 -> 23.3; fp16, B1 H8 N2048 D128 67.4 -> 58.5).  The rings of a
// D >= 64 workgroup fill a CU's LDS whatever its rows, so from 129 on the halves take a second round (bf16, B1 H9 N2048 D64
// 38.3 -> 56.8, B1 H12 N2048 D64 41.4 -> 56.9, D128 75 -> 105); at D32 two share a CU and take turns (fp16, B1 H9 N2048 28.4 ->
// 30.3, 256 blocks of N = 512 11.1 -> 11.6).
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

// Whether a backward goes into one grid (bwd_pair_kernel) instead of a dK/dV and a dQ launch.  `n`, `blocks`: as above;
// `stages`: what is asked for (4 dK/dV, 8 dQ).
// At D = 128 always: its dQ blocks are four waves at one wave per SIMD either way.  At D <= 64 the dQ kernel of its own has
// eight waves and 256 rows, two waves per SIMD, and is the faster one on a full chip (headline size: 437 us against 510), so
// it is a matter of rounds.  Microseconds per round of 256 workgroups at N = 2048, D = 64, which scale alike with N and D:
// 79 for key blocks, 64 for query blocks of the one grid, 109 for 256-row blocks of the dQ kernel; a grid that is dealt from
// one list ends with a partial round of 25.  Measured over N = 128 ... 4096 and 192 ... 1280 blocks: gains of up to 24 % on
// the line's near side, up to 6 % on its far side, 7 % in padded sequences.
// Causal blocks differ in length and fill the rounds by themselves: the one grid is faster below 576 blocks
// (by 5 % at 512, 40 % at 256) and slower above 640 (by 2-5 %).  Those of a unit of one or two blocks hardly differ: at N = 256
// the rounds decide as without a mask (us of the whole backward, two launches -> one grid: D64 512 blocks 71 -> 74, 640
// blocks 95 -> 86, D32 640 blocks 61 -> 55); at N = 128 there is one key block and one query block to a unit, and two launches
// are ahead from 448 blocks on (D32, 448 blocks 36 -> 39, 512 blocks 40 -> 42; 384 blocks 34 -> 32).
constexpr bool bwd_one_grid(int d, bool dropout, bool causal, int n, long long blocks, unsigned stages) {
  if (dropout) return false;          // the dropout instantiations are not pipelined
  if (d == 128) return true;
  const bool wide = n % 256 == 0;     // the dQ kernel of its own has its 256-row blocks
  // n an odd multiple of 128: its 128-row variant has one wave per SIMD at D = 64 (LDS), and this one is pipelined
  if (d == 64 && !wide && (stages & 8u)) return true;
  if ((stages & 12u) != 12u) return blocks <= kNumCU;
  if (causal && n > 256) return blocks <= 576;
  if (causal && n == 128) return blocks <= 384;
  const long long two = 79 * ((blocks + 255) / 256) + 109 * ((blocks + 511) / 512);
  const long long one = (d == 32 ? 150 : 143) * blocks / 256 + 25;
  return one < two;
}

// A weight gradient of the layer (wgrad_kernel, layer.hip): workgroups per 128 x 128 tile and the 64-token slabs that each
// of them takes.  `tiles`: of all the weights of the launch.  One workgroup fills a CU's LDS, so tiles are split as far as one
// round of workgroups goes, but not below four slabs, where starting a workgroup and adding its sums takes longer than they do.
constexpr int kWgradTile = 128, kWgradSlab = 64;
struct WgradSplit { int splits, slabs; };
constexpr WgradSplit wgrad_split(long long tiles, int tokens) {
  const int all = (tokens + kWgradSlab - 1) / kWgradSlab;
  long long want = kNumCU / tiles;
  if (want > all / 4) want = all / 4;
  if (want < 1) want = 1;
  const int slabs = (int)((all + want - 1) / want);
  return {(all + slabs - 1) / slabs, slabs};
}

}  // namespace da_abi
