// The launch geometries of a forward and of a backward as pure functions of the sizes and options.  Plain C++: a test
// compiles it by itself.
#pragma once

namespace da_abi {

constexpr int kNumCU = 256;

// Whether a forward runs in 64-row, four-wave workgroups instead of 128-row ones.  (The reference autotunes its tiles per
// (N, D, Dv), src/kernel.py:12-19; there is no tuning state here.)  `n`: the padded sequence length, a multiple of 128;
// `blocks`: B*H*n/128.  Figures: us of a launch, 128-row -> 64-row.  (The lines were taken before P*V ran one tile behind in D = 32 and in
// 64-row blocks at D = 64.  Measured again since, at 52 pairs about them, each takes the side that is ahead: D32 B1 H9 N2048 26.4 -> 27.3,
// 256 causal blocks of N = 128 8.0 -> 7.8; D64 B1 H8 N2048 39.2 -> 30.1, B1 H9 39.9 -> 53.1.)
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
// the line's near side, up to 6 % on its far side, 7 % in padded sequences; again with the key blocks' requests across steps, at 37 pairs
// about the lines: two launches over one grid within 0.04 of what it was.
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

// Whether the layer's three input projections, or their input gradient, are one product with the three weights E x E copied
// one behind another, instead of a product for each.  One product of 3E fills the chip where one of E does not, and saves two
// launches; the copy moves 12 E^2 bytes, and a product on few tokens is bound by the 6 E^2 that it reads.  Device time of
// both, us, fp16 (bf16 the same within 10 %, with the weights of several layers in turn), one product | three:
//   E 1024, 77 tokens 15 | 19, 1024 22 | 30, 8192 66 | 70;  E 2048: 24 | 29, 40 | 51, 164 | 162;  E 3584: 45 | 58, 94 | 110
//   E 4096, 32 tokens 50 | 37, 77 54 | 48, 128 56 | 69, 512 83 | 91, 1024 117 | 129, 4096 322 | 299
//   E 5120, 32 tokens 82 | 57, 77 89 | 65, 128 91 | 100, 512 129 | 147, 1024 189 | 197, 4096 528 | 576
//   E 5632, 32 tokens 115 | 61, 512 167 | 147, 2048 489 | 338, 4096 712 | 661;  E 8192: 229 | 96, 299 | 249, 697 | 594, 1238 | 1130
// Up to E 4730 the weights and their copy fit the last-level cache of 256 MB, up to E 5120 most of them do; beyond that both
// go to memory.  Few tokens at E 4096 to 4608: the three products are the faster ones on the device, but 37 us more of host
// time, which is what bounds such a call (E 4096, 77 tokens, the layer's forward: 66 us on the device instead of 75, and 102
// us a call instead of 74; E 5120 77 instead of 123, and 101 instead of 122; E 8192 171 instead of 282 both ways).  At E 3072 to
// 4096 the single product of many tokens takes a worse library kernel (E 3072, 4096 tokens 216 | 206, 8192 466 | 406; not at E
// 2560 and from 4608 on).  The input gradient (E 2048, 77 tokens 32 | 34, 4096 110 | 138; E 4096 81 | 68, 353 | 400; E 7168 280 |
// 162, 1446 | 1111; E 8192 320 | 175, 1382 | 1396) has no such line, and its call with few tokens is bound by host time further up.
constexpr bool layer_packed(bool backward, long long E, long long tokens) {
  if (E > 5120) return false;
  return backward || !((E > 4608 && tokens <= 96) || (E >= 3072 && E <= 4096 && tokens >= 4096));
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

// Whether a layer's weight gradients go to wgrad_kernel, in one launch, or are a library product each.  The library's tiles
// for few outputs and a long contraction leave most of the chip idle; from E 2560 on its larger tiles fill the chip and read
// less.  Device time, us, fp16, library | kernel with the sum of its splits:
//   four weights: E 256, 77 tokens 52 | 9, 8192 190 | 19;  E 512 23 | 9, 204 | 31;  E 768 23 | 9, 198 | 61;  E 1024 23 | 10, 212 | 73
//     (946 TFLOP/s), 16384 403 | 141;  E 1152 28 | 16, 243 | 147;  E 1280 28 | 17, 257 | 132;  E 1536 34 | 23, 323 | 202;
//     E 1792 35 | 29, 311 | 266;  E 2048 36 | 30, 337 | 296, 16384 686 | 637;  E 2560 45 | 47, 2048 143 | 156, 8192 480 | 516 (16384
//     1494 | 1028);  E 3072 56 | 59, 638 | 722;  E 4096 68 | 102, 961 | 1308
//   one weight: E 384, 256 tokens 7.0 | 8.7, 1000 14.0 | 12.3;  E 512, 77 tokens 6.7 | 8.6, 2048 17 | 15, 8192 52 | 23, 16384 98 | 23;
//     E 768, 1000 tokens 14.3 | 15.6, 2048 17.2 | 18.2, 4096 29 | 22;  E 1024, 77 tokens 7.0 | 8.6, 1000 14.5 | 20.8, 2048 17.6 |
//     22.7, 4096 31 | 24, 8192 56 | 30;  E 1152, 2048 tokens 21.7 | 23.4, 4096 34 | 33;  E 1280, 1000 tokens 17.5 | 20.3, 2048
//     21.7 | 21.1;  E 1536, 77 tokens 9.6 | 9.0, 1000 21.0 | 15.4;  two weights: the kernel throughout (E 512, 77 tokens 12 | 9)
// A single short product is a library tile to each CU and no splits to add, while the kernel's are few tiles, split.
constexpr bool wgrad_own(int weights, long long E, long long tokens) {
  if (E % kWgradTile != 0 || E > 2048) return false;
  return weights > 1 || E <= 256 || E >= 1536 || tokens > 2 * E;
}

}  // namespace da_abi
