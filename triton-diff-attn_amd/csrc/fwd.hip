// Differential-attention forward for gfx950: two online-softmax streams per query row, fused
// lambda-combine and RMSNorm epilogue.  Computes what the reference's forward kernel computes
// (src/kernel.py:20-207) with a different decomposition:
//
//   * a workgroup of 8 waves owns 128 query rows (4 waves and 64 rows for small grids); waves 0-3 run softmax stream 1 (Q1,K1) and
//     waves 4-7 run stream 2 (Q2,K2) for the same rows, 32 rows per wave.  All 8 waves share
//     the K1/K2/V tiles, double-buffered in LDS, and the two streams meet only in the epilogue;
//   * scores are computed transposed, S^T = K * Q^T (K fragments from LDS as the MFMA A operand,
//     Q fragments resident in registers as B), so each lane owns one query column: the row
//     max / row sum are in-lane reductions plus one exchange with lane^32, and the rescale
//     factor, 1/l, lambda-combine and RMSNorm are per-lane scalars;
//   * the P^T accumulator registers are reused directly (after fp16 packing) as the B operand of
//     O^T = V^T * P^T; the V^T A-fragments come from the row-major V tile through the
//     transposing LDS read, using the same key permutation as the accumulator layout.
#include <type_traits>

#include "dispatch.hpp"
#include "params.hpp"

namespace DA_NS {

// SMALL: 64 query rows per workgroup (four waves), for problems whose 128-row blocks leave much of the chip idle and
// for the D = 128 instantiations with dropout, which do not fit the register budget of two waves per SIMD.
template <int D, bool SMALL = false>
struct FwdCfg {
  static constexpr int DV = 2 * D;
  static constexpr int BN = (D <= 64) ? 64 : 32;   // keys per tile
  static constexpr int QS = 1;                     // 32-row query blocks per wave
  // query rows per workgroup
  static constexpr int BM = SMALL ? 64 : 128;
  static constexpr int NW = 2 * BM / (32 * QS);    // waves per workgroup: half of them per softmax stream
  static constexpr int NT = NW * 64;
  // waves per SIMD the register budget is sized for: two, except in the four-wave D = 128 workgroups, whose
  // dropout instantiations need more than 256 registers
  static constexpr int OCC = (D == 128 && SMALL) ? 1 : 2;
  // thread count the register budget is derived from: with fewer than 4 * OCC waves in a workgroup the
  // occupancy attribute alone does not hold the allocator to 512 / OCC registers (the four-wave variant at
  // D = 64 then took 336 and shuffled values between the two halves of the register file all through its loop)
  static constexpr int REG_NT = (OCC * 256 > NT) ? OCC * 256 : NT;
  static constexpr int K_TILE = BN * D;            // halfs, one stream (swizzled, unpadded)
  static constexpr int V_TILE = BN * DV;
  static constexpr int K_BUF = 2 * K_TILE;         // K1 and K2 of one tile
  // Ring depth.  The loop is unrolled over one turn of the ring with every buffer known at compile time: an LDS address is then a
  // per-lane register plus an immediate offset, with no arithmetic inside the loop.  Where the workgroup meets every second tile all
  // four buffers are in use (in one iteration and the next, K tiles t+1 and t+2 are read while t+3 and t+4 arrive, V tiles t-1 and t, or t and
  // t+1, while the next two do); where it meets every tile three would do.
  static constexpr int NBUF = 4;
  // A barrier every second tile instead of every tile (the ring allows it): measured in one GPU call,
  // 3.3 % faster at D = 32, 3 % slower at D = 64 and 5 % slower at D = 128.  In the 64-row workgroups at D = 64, whose waves have a
  // SIMD each, it is the faster one, too (causal, B1 H4 N8192 124.4 -> 122.2 us, B1 H8 N2048 32.8 -> 31.6).
  static constexpr bool PAIR = (D == 32 || (D == 64 && SMALL));
  static constexpr int KBUF_BYTES = K_BUF * 2, VBUF_BYTES = V_TILE * 2, VBASE_BYTES = NBUF * KBUF_BYTES;
  static_assert(NBUF * KBUF_BYTES <= 65536 && NBUF * VBUF_BYTES <= 65536, "immediate offsets reach every buffer");
  static constexpr int TILES = NBUF * (K_BUF + V_TILE);
  // halfs needed by the epilogue: per pair of waves (stream 1, stream 2 of the same 32 rows) an fp32 exchange
  // block of 32 x DV values, which the stream-1 wave reuses for its staged rows, and the staging block
  // (32 rows of DV + 8 halfs) of the stream-2 wave
  // (a block holds the exchange, and after it has been read the staged rows of both waves of the pair)
  static constexpr int XCH_BLOCK = (64 * DV > 2 * 32 * (DV + 8)) ? 64 * DV : 2 * 32 * (DV + 8);
  static constexpr int XCHG = (NW / 2) * XCH_BLOCK;
  static constexpr int SMEM = (TILES > XCHG) ? TILES : XCHG;
};

constexpr float kRescaleThreshold = 8.0f;   // log2 units: probabilities stay below 2^8 between updates of the row max
constexpr float kRescaleSum = 16384.0f;     // of late_iteration: a lane's share of a tile's row sum, which no probability of it exceeds, between those updates
constexpr float kRescaleWatch = 14.0f;      // log2 units, of a watching late_iteration: no probability there exceeds 2^14
constexpr int kWatchMoves = 3;              // moves in a turn of four tiles that make a wave watch

// MASK: 0 none; 1 causal (key <= query); 2 the last keys of the sequence are padding (key < n_keys).
// With the causal mask the padding needs no extra test: a padded key lies after every real query.
// DROP: dropout on both softmax maps (not in the reference, which lists it as missing,
// src/kernel.py:4): a dropped probability still counts in its row's sum but not in P*V, and the
// kept ones are scaled by 1/(1-p) -- in the epilogue, together with 1/l.
template <int D, bool RMS, int MASK, bool DROP, bool SMALL = false>
__global__ __launch_bounds__((FwdCfg<D, SMALL>::REG_NT)) __attribute__((amdgpu_waves_per_eu(FwdCfg<D, SMALL>::OCC, FwdCfg<D, SMALL>::OCC)))
void fwd_kernel(FwdParams p) {
  using C = FwdCfg<D, SMALL>;
  constexpr int DV = C::DV, BN = C::BN, NW = C::NW, BM = C::BM, QS = C::QS;
  constexpr int NKS = D / 16;                // k-steps of the score product
  constexpr int NKT = BN / 32;               // 32-key tiles of S^T
  constexpr int NKK = BN / 16;               // k-steps of the P*V product
  constexpr int NOT = DV / 32;               // 32-row tiles of O^T

  __shared__ __attribute__((aligned(16))) half_t smem[C::SMEM];
  lds_half* const sKbuf = (lds_half*)smem;                 // [NBUF][K1 tile, K2 tile]
  lds_half* const sVbuf = sKbuf + C::NBUF * C::K_BUF;      // [NBUF][V tile]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int st = wave / (NW / 2), qw = wave % (NW / 2);   // stream, block of 32*QS rows inside the workgroup
  const int j = lane & 31, g = lane >> 5;

  const int n_qt = p.N / BM;
  constexpr bool CAUSAL = (MASK == 1), PADDED = (MASK == 2);
  // rows past the real length are neither read from the caller's tensors nor written to y: checked in both
  // masked variants (the causal one serves padded sequences too), compiled out of the plain one
  constexpr bool TAIL = (MASK != 0);
  // the masked loop of the 128-row D = 128 workgroup has no register to spare (see the iteration)
  constexpr bool kLean = TAIL && D == 128 && !SMALL;
  // P*V runs one tile behind the exponentials (late_iteration).  (The causal 64-row workgroup at D = 64 went to scratch that way.)
  constexpr bool kLate = D == 32 || (D == 64 && SMALL && MASK != 1);
  constexpr bool kWatch = D == 32;      // with watching iterations
  int bh, qt;
  if constexpr (CAUSAL) {   // the last query block of a unit sees the most keys
    const UnitBlock ub = longest_first(blockIdx.x, p.BH);
    bh = ub.unit; qt = n_qt - 1 - ub.rank;
  } else {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    bh = tile / n_qt; qt = tile % n_qt;
  }
  // element offsets of the unit's first row and the row strides of its tensors
  const size_t qk_base = da_abi::unit_base(p, p.sqk, bh);
  const size_t v_base = da_abi::unit_base(p, p.sv, bh);
  const int qk_n = (int)p.sqk.n, v_n = (int)p.sv.n;
  const int qrow0 = qt * BM + qw * 32 * QS + j;   // this lane's query row of block qs is qrow0 + 32*qs
  // used with dropout only: hash key of this wave's softmax stream, the counter of this query's first key pair, the
  // counters' lane-dependent low bits, and what a block of eight keys adds inside a tile
  const DropoutKey dkey = dropout_key(p.drop, 2u * bh + st);
  const unsigned hrow = (unsigned)(qrow0 >> 1) * ((unsigned)p.N / 2), hlow = (unsigned)(2 * g + (qrow0 & 1));
  const DropoutSel dsel = dropout_sel_query(qrow0 & 1);
  unsigned hstep[BN / 8];
#pragma unroll
  for (int v = 0; v < BN / 8; ++v) hstep[v] = dropout_window_step<BN / 2>(dkey, v);

  // Asked for here, with the first tiles: behind the loop its latency would be in nobody's shadow.
  const float lam_load = da_abi::lambda_of_unit(p, bh);

  // Q fragments (B operand): column j = this lane's query, k = 8g..8g+7 of each 16-wide k-step.
  // They are pre-multiplied by sm_scale*log2(e), so the MFMA result is the score in log2 units.
  h8 qf[QS][NKS];
  {
    const float c = p.sm_scale * kLog2e;
#pragma unroll
    for (int qs = 0; qs < QS; ++qs) {
      // a padding row (past the sequence's real length) stands in with the last real row: finite scores,
      // results that are never stored
      int qr = qrow0 + 32 * qs;
      if (TAIL && qr >= p.n_keys) qr = p.n_keys - 1;
      const half_t* r = (st ? p.q2 : p.q1) + qk_base + (size_t)qr * qk_n + 8 * g;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        h8 q = *reinterpret_cast<const h8*>(r + 16 * ks);
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = (half_t)((float)q[e] * c);
        qf[qs][ks] = q;
      }
    }
  }

  f16v o[QS][NOT];
#pragma unroll
  for (int qs = 0; qs < QS; ++qs)
#pragma unroll
    for (int t = 0; t < NOT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[qs][t][r] = 0.f;
  // The running reference m of the online softmax is folded into the score product as the
  // initial accumulator value -m, so the MFMA result is already s - m.
  float m[QS], l[QS];
  f16v negm[QS];
#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    m[qs] = 0.f; l[qs] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) negm[qs][r] = 0.f;
    asm volatile("" : "+v"(negm[qs]));   // sixteen registers of its own: the score products take it as their C operand as it is
  }

  using KTile = AsyncTile<BN, D, NW>;
  using VTile = AsyncTile<BN, DV, NW>;
  const half_t* gk1 = p.k1 + qk_base;
  const half_t* gk2 = p.k2 + qk_base;
  const half_t* gv = p.v + v_base;
  // causal: keys beyond the last row of the workgroup are visited only to make the tile count even (64-row
  // workgroups with 64-key tiles: every other one has a last tile that is masked throughout; N is a multiple of 128)
  const int n_tiles = CAUSAL ? ((qt + 1) * (BM / BN) + 1) & ~1 : p.N / BN;
  constexpr int VH = (VTile::PER + 1) / 2;   // V instructions are issued in two groups
  const unsigned k_off = KTile::lane_off(wave, lane, qk_n), v_off = VTile::lane_off(wave, lane, v_n);
  auto tail_lane = [&] { return kLean ? lane_again() : lane; };
  // With padding, the tiles that reach past the last real row are copied with their row index clamped to it.
  // `tail` (a compile-time tag) says whether the call site can meet such a tile at all.  Where P*V runs late every copy of such a call site is
  // clamped: the four branches of an iteration cut its interleaved products apart and cost more than the eight instructions.  us,
  // fp16, with them -> without: D32 H8 N1000 12.6 -> 12.1, causal 13.0 -> 12.4, H16 N77 5.45 -> 5.11, causal N512 9.4 -> 9.0; D64 H16 N77 7.6 ->
  // 7.1, H8 N1000 18.4 -> 17.9; with dropout 8.6 -> 8.1.
  auto load_k1 = [&](int tk, int buf, auto tail) DA_INLINE {
    if (TAIL && decltype(tail)::value && (kLean || kLate || (tk + 1) * BN > p.n_keys))
      KTile::template issue_clamped<0, KTile::PER, kLean>(gk1 + (size_t)tk * BN * qk_n, sKbuf + buf * C::K_BUF, wave, tail_lane(), k_off, qk_n,
                                                          p.n_keys - 1 - tk * BN);
    else
      KTile::issue_at(gk1 + (size_t)tk * BN * qk_n, sKbuf + buf * C::K_BUF, wave, lane, k_off, qk_n);
  };
  auto load_k2 = [&](int tk, int buf, auto tail) DA_INLINE {
    if (TAIL && decltype(tail)::value && (kLean || kLate || (tk + 1) * BN > p.n_keys))
      KTile::template issue_clamped<0, KTile::PER, kLean>(gk2 + (size_t)tk * BN * qk_n, sKbuf + buf * C::K_BUF + C::K_TILE, wave, tail_lane(), k_off,
                                                          qk_n, p.n_keys - 1 - tk * BN);
    else
      KTile::issue_at(gk2 + (size_t)tk * BN * qk_n, sKbuf + buf * C::K_BUF + C::K_TILE, wave, lane, k_off, qk_n);
  };
  auto load_va = [&](int tv, int buf, auto tail) DA_INLINE {
    if (TAIL && decltype(tail)::value && (kLean || kLate || (tv + 1) * BN > p.n_keys))
      VTile::template issue_clamped<0, VH, kLean>(gv + (size_t)tv * BN * v_n, sVbuf + buf * C::V_TILE, wave, tail_lane(), v_off, v_n, p.n_keys - 1 - tv * BN);
    else
      VTile::template issue_at<0, VH>(gv + (size_t)tv * BN * v_n, sVbuf + buf * C::V_TILE, wave, lane, v_off, v_n);
  };
  auto load_vb = [&](int tv, int buf, auto tail) DA_INLINE {
    if (TAIL && decltype(tail)::value && (kLean || kLate || (tv + 1) * BN > p.n_keys))
      VTile::template issue_clamped<VH, VTile::PER, kLean>(gv + (size_t)tv * BN * v_n, sVbuf + buf * C::V_TILE, wave, tail_lane(), v_off, v_n, p.n_keys - 1 - tv * BN);
    else
      VTile::template issue_at<VH, VTile::PER>(gv + (size_t)tv * BN * v_n, sVbuf + buf * C::V_TILE, wave, lane, v_off, v_n);
  };
  constexpr std::true_type with_tail{};
  constexpr std::false_type no_tail{};

  // Per-lane LDS byte addresses, computed once.  The XOR swizzle makes the address of a fragment a
  // different function of the lane for every 16-byte chunk column, so there is one register per chunk
  // column a lane reads; the ring buffer, the 32-key block and the k-step of 16 keys are multiples of 16
  // rows, which the swizzle does not see, and travel in the instructions' immediate offsets.
  // transposing-read coordinates of this lane inside a 16-key k-step: key row and feature column
  const int tr_row = 4 * g + ((lane & 15) >> 2);
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const unsigned lds0 = (unsigned)(unsigned long)((DA_LDS char*)smem);
  unsigned kb[NKS], vtr[NOT][2];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) kb[ks] = lds0 + 2u * (unsigned)(st * C::K_TILE + swz_off<D>(j, 16 * ks + 8 * g));
#pragma unroll
  for (int tt = 0; tt < NOT; ++tt)
#pragma unroll
    for (int e = 0; e < 2; ++e) vtr[tt][e] = lds0 + C::VBASE_BYTES + 2u * (unsigned)swz_off<DV>(tr_row + 8 * e, 32 * tt + tr_col);
  // kept as they are: the compiler neither folds constants into them nor recomputes them in the loop
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(kb[ks]));
#pragma unroll
  for (int tt = 0; tt < NOT; ++tt) asm volatile("" : "+v"(vtr[tt][0]), "+v"(vtr[tt][1]));

  // A-fragments of K for all k-steps of all 32-key tiles: row kt*32 + j, halfs 16ks + 8g .. +7
  auto read_k = [&](int byte_off, h8 (&ka)[NKT][NKS]) {
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) ka[kt][ks] = lds_read_at<h8>(kb[ks], byte_off + kt * 32 * D * 2);
  };
  // Score products number I0 .. I1-1 of a tile, counted in issue order: 32-key tile kt, k-step ks is number
  // kt * NKS + ks.  The first product of a 32-key tile starts from the running reference.
  auto scores_of = [&](const h8 (&ka)[NKT][NKS], f16v (&s)[QS][NKT], auto i0, auto i1) DA_INLINE {
#pragma unroll
    for (int i = decltype(i0)::value; i < decltype(i1)::value; ++i) {
      const int kt = i / NKS, ks = i % NKS;
#pragma unroll
      for (int qs = 0; qs < QS; ++qs) {
        if (ks == 0) s[qs][kt] = negm[qs];
        s[qs][kt] = mfma32(ka[kt][ks], qf[qs][ks], s[qs][kt]);
      }
    }
  };
  constexpr int NSC = NKT * NKS;      // score products per tile and 32-row block
  auto scores = [&](const h8 (&ka)[NKT][NKS], f16v (&s)[QS][NKT]) {
    scores_of(ka, s, std::integral_constant<int, 0>{}, std::integral_constant<int, NSC>{});
  };
  // How many of the next tile's score products are issued ahead of the row maxima of this one; the rest follow
  // the reference update and run under the first exponentials, which have no other matrix work beside them.
  // The split is between 32-key tiles (D = 32 has late_iteration and no split).  Measured against all of them ahead, inside one GPU
  // call each: the first of two tiles ahead -2.5 % at D = 64 (0.442 -> 0.432 ms); none ahead the same at
  // D = 64 and +0.7 % at D = 128; a D = 128 tile is a single 32-key tile, and splitting it in the middle
  // of its k-steps cost 1.5 %, so it stays whole and ahead.
  constexpr int SC_EARLY = DROP ? NSC : ((NKT + 1) / 2) * NKS;
  constexpr int KT_EARLY = (SC_EARLY + NKS - 1) / NKS;     // 32-key tiles whose first product is among them
  constexpr std::integral_constant<int, 0> sc_first{};
  constexpr std::integral_constant<int, SC_EARLY> sc_split{};
  constexpr std::integral_constant<int, NSC> sc_end{};

  // loads this wave issues per iteration (one K1, one K2 and one V tile)
  const int loads_per_iter = 2 * KTile::count(wave) + VTile::count(wave);
  auto clampt = [&](int t) { return t < n_tiles ? t : n_tiles - 1; };   // past the end: harmless re-reads

  // The loop below runs whole turns of the ring (NBUF iterations); the tile count is even, so when it is
  // not a multiple of four, half a turn comes first and tile 0 goes into buffer 2: tile t is in buffer
  // (t + b0) % NBUF, b0 = 0 or 2.
  static_assert(C::NBUF == 4, "the loop is unrolled over a ring of four");
  const bool head_half = (n_tiles & 2) != 0;
  const int b0 = head_half ? 2 : 0;
  // prologue: K tiles 0..2 and V tiles 0..1; scores of tile 0
  load_k1(0, b0, with_tail); load_k2(0, b0, with_tail); load_va(0, b0, with_tail); load_vb(0, b0, with_tail);
  load_k1(clampt(1), b0 + 1, with_tail); load_k2(clampt(1), b0 + 1, with_tail);
  if (!kLate || head_half) { load_va(clampt(1), b0 + 1, with_tail); load_vb(clampt(1), b0 + 1, with_tail); }
  if (n_tiles > 2) { load_k1(2, (b0 + 2) % 4, with_tail); load_k2(2, (b0 + 2) % 4, with_tail); }
  if constexpr (kLate) {
    // the V tile in front of the first one, which the loop's first iteration multiplies with zero probabilities
    if (!head_half) {
      DA_LDS u32x4* z = (DA_LDS u32x4*)(sVbuf + 3 * C::V_TILE);
      for (int k = tid; k < C::V_TILE / 8; k += C::NT) z[k] = u32x4{0u, 0u, 0u, 0u};
    }
  }
  wait_async_tiles();
  const float lam = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, lam_load)));
  __syncthreads();
  // Keys past the diagonal, or past the last real key, are masked: `rel` is the last visible key minus the key
  // index of register 0, tile 0
  auto mask_scores = [&](f16v (&s)[QS][NKT], int rel) DA_INLINE {
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[0][kt][r] = (kt * 32 + 8 * (r / 4) + (r % 4) > rel) ? -INFINITY : s[0][kt][r];
  };
  // the largest score of this lane
  auto lane_max = [&](const f16v (&s)[NKT]) DA_INLINE {
    float mx0 = fmaxf(s[0][0], s[0][1]), mx1 = fmaxf(s[0][2], s[0][3]);
    float mx2 = fmaxf(s[0][4], s[0][5]), mx3 = fmaxf(s[0][6], s[0][7]);
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int r = (kt == 0 ? 8 : 0); r < 16; r += 8) {
        mx0 = fmaxf(mx0, fmaxf(s[kt][r + 0], s[kt][r + 1]));
        mx1 = fmaxf(mx1, fmaxf(s[kt][r + 2], s[kt][r + 3]));
        mx2 = fmaxf(mx2, fmaxf(s[kt][r + 4], s[kt][r + 5]));
        mx3 = fmaxf(mx3, fmaxf(s[kt][r + 6], s[kt][r + 7]));
      }
    return fmaxf(fmaxf(mx0, mx1), fmaxf(mx2, mx3));
  };
  constexpr int NPV = NKK * NOT;
  auto vt_frag_at = [&](int i, int voff) DA_INLINE {
    const int kk = i / NOT, tt = i % NOT;
    return join(lds_read_tr_at(vtr[tt][0], voff + 16 * kk * DV * 2), lds_read_tr_at(vtr[tt][1], voff + 16 * kk * DV * 2));
  };
  constexpr int KA = 4, VA = 3;              // K and V^T fragments requested ahead of their products
  h8 kfirst[KA], vfirst[VA];                 // the first ones of the next iteration
  auto k_frag_at = [&](int i, int koff) DA_INLINE { return lds_read_at<h8>(kb[i % NKS], koff + (i / NKS) * 32 * D * 2); };
  auto request_first_k = [&](int koff) DA_INLINE {
#pragma unroll
    for (int i = 0; i < KA && i < NSC; ++i) kfirst[i] = k_frag_at(i, koff);
  };
  auto request_first = [&](int koff, int voff) DA_INLINE {
    request_first_k(koff);
#pragma unroll
    for (int i = 0; i < VA; ++i) vfirst[i] = vt_frag_at(i, voff);
  };
  int moves = 0;           // kWatch: how often the reference moved in this turn of the ring
  f16v s_a[QS][NKT], s_b[QS][NKT];
  {
    h8 ka[NKT][NKS];
    if (head_half) read_k(2 * C::KBUF_BYTES, ka);
    else read_k(0, ka);
    scores(ka, s_a);
  }
  if constexpr (kLate) {
    if (head_half) request_first_k(3 * C::KBUF_BYTES);
    else request_first(1 * C::KBUF_BYTES, 3 * C::VBUF_BYTES);
  }
  // P of the tile in front of the current one
  u32x4 pw[NKK];
  if constexpr (kLate) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) pw[kk] = u32x4{0u, 0u, 0u, 0u};
    // the first tile's row maxima are the reference to begin with
    if constexpr (TAIL) {
      if (BN > (CAUSAL ? qt * BM + qw * 32 + 1 : p.n_keys)) mask_scores(s_a, (CAUSAL ? qt * BM + qw * 32 + j : p.n_keys - 1) - 4 * g);
    }
    m[0] = pair_max(lane_max(s_a[0]));
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int r = 0; r < 16; ++r) s_a[0][kt][r] -= m[0];
#pragma unroll
    for (int r = 0; r < 16; ++r) negm[0][r] = -m[0];
    asm volatile("" : "+v"(negm[0]));
  }
  enum Kind { kFollows, kOpens, kWatches };
  // One iteration at D = 32, where the vector instructions of a tile take longer than its matrix instructions and the two waves of
  // a SIMD leave each barrier in step, and of the 64-row workgroups at D = 64, which have one wave to a SIMD: the exponentials of tile t,
  // the score product of tile t+1 and the P*V product of tile t-1, none of which depends on another, interleaved in one basic block.
  // Row maxima are formed for the first tile only: the row sum of the rounded probabilities, which is formed anyway, says afterwards
  // whether they left the range of the 16-bit type with room to spare, and then this tile's are formed again.  The first fragments of an
  // iteration are requested in the one before it, or where the workgroup meets between them right behind the meeting.  K tile t+3 goes
  // to the buffer of tile t-1, whose scores were formed two iterations ago, V tile t+1 to that of tile t-3, multiplied two
  // iterations ago; the one meeting in two iterations lies in between.
  // fp16, us, before -> now: D32 B4 H32 N2048 277 -> 259, B1 H16 N16384 1903 -> 1786, B1 H2 N4096 37.0 -> 31.5, B1 H8 N2048 22.5 -> 20.2;
  // D64 in 64-row workgroups B1 H8 N2048 37.3 -> 35.3, N2000 38.8 -> 36.3, B1 H4 N1000 19.3 -> 18.0, B1 H16 N512 11.9 -> 11.4.  Not for
  // the 128-row workgroups at D = 64, which are bound by power (1.7 GHz of 2.4: 425 us both ways at B4 H32 N2048), nor at D = 128,
  // where it spills.
  // `kind`: what the iteration leaves out or looks for.
  // kWatches (D = 32): scores that move the reference at one tile may do so at most of them, and to form a tile's probabilities a second
  // time takes half as long as a tile.  Behind a turn of the ring with three such moves a wave goes on with iterations that look at
  // the row maxima ahead of the exponentials, where a move costs no second ones.  (A look in every iteration, behind a branch, cost
  // small grids whose reference never moves 1 to 4 %; a way back to the first kind of iteration went to scratch; at two moves a turn
  // scores with a deviation of 4 to 6 lose 5 %, at four the gain is half.)  us, fp16, scores of a standard deviation of 1, 6, 9, 16 and
  // 36, row maxima at every tile (`iteration`) | never, probabilities a second time | now:
  //   B4 H16 N2048  126 133 136 142 147 | 122 130 143 165 186 | 120 131 146 153 151;  causal 78 82 86 89 91 | 76 82 90 103 112 | 75 83 91 96 95
  //   B1 H8 N2048  23.4 24.4 25.2 26.1 26.5 | 20.3 23.0 25.4 28.5 30.2 | 20.2 23.4 25.8 27.0 26.7;  N8192 230 228 226 235 245 | 216 221 227 249 279 |
  //   216 223 241 255 251;  scores that grow by 14 powers of two a tile, B4 H16 N2048 157 | 203 | 164
  // Not at D = 64, where the second loop costs launches whose reference never moves more (H16 N256 8.25 -> 8.42, N512 11.05 -> 11.23) than
  // such scores are worth: B1 H8 N2048, deviation of 9 and 16, 35.1 35.9 | 35.4 39.5, with it 35.2 36.5; sequences of up to four tiles
  // have no second turn (N256, deviation of 16, 9.1 | 9.7).
  // kOpens: the first iteration where half a turn comes first, which is compiled by itself: there is no product to make up for, V
  // tile 1 was requested with the first tiles, and the scores are masked.  With them it cost sequences of up to 128 keys, which
  // have no other iterations to win it back in, 2 to 7 % against
  // the loop this one replaced (`iteration`); us, fp16, that loop -> with them -> now: D32 H16 N77 causal 6.25 -> 6.67 -> 6.07, N128 causal
  // 5.87 -> 6.22 -> 5.77, D64 H16 N77 8.07 -> 8.27 -> 7.77, N128 6.51 -> 6.60 -> 6.39 (with dropout 7.10 -> 7.29 -> 7.20).
  auto late_iteration = [&](int t, auto pos_tag, auto tail, auto kind, f16v (&s_cur)[QS][NKT], f16v (&s_nxt)[QS][NKT]) DA_INLINE {
    constexpr int POS = decltype(pos_tag)::value;
    constexpr bool kOpening = decltype(kind)::value == kOpens, kWatching = decltype(kind)::value == kWatches;
    constexpr int KR = (POS + 1) % 4, KP = (POS + 3) % 4, VR = (POS + 3) % 4, VP = (POS + 1) % 4;
    constexpr int VOFF = VR * C::VBUF_BYTES, KOFF = KR * C::KBUF_BYTES;
    const int tk = clampt(t + 3), tv = clampt(t + 1);
    constexpr bool kTail = TAIL && decltype(tail)::value;
    load_k1(tk, KP, tail);
    h8 ka[NSC], vfr[NPV];
    if constexpr (!kOpening) {
#pragma unroll
      for (int i = 0; i < VA; ++i) vfr[i] = vfirst[i];
    }
#pragma unroll
    for (int i = 0; i < KA && i < NSC; ++i) ka[i] = kfirst[i];
    if constexpr (kTail && !kOpening) {
      if ((t + 1) * BN > (CAUSAL ? qt * BM + qw * 32 + 1 : p.n_keys))
        mask_scores(s_cur, (CAUSAL ? qt * BM + qw * 32 + j : p.n_keys - 1) - t * BN - 4 * g);
    }
    // The reference moves up by d.  P*V of the tiles in front of this one is complete at the end of the iteration only, where
    // `lower` brings it and the row sum to the new reference.
    float d = 0.f;
    auto raise = [&](float largest) DA_INLINE {
      d = fmaxf(pair_max(largest), 0.f);
      m[0] += d;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) s_cur[0][kt][r] -= d;
#pragma unroll
      for (int r = 0; r < 16; ++r) negm[0][r] = -m[0];
      asm volatile("" : "+v"(negm[0]));
    };
    auto lower = [&]() DA_INLINE {
      const float alpha = fast_exp2(-d);
      l[0] *= alpha;
#pragma unroll
      for (int tt = 0; tt < NOT; ++tt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[0][tt][r] *= alpha;
    };
    bool moved = false;
    if constexpr (kWatching) {
      const float largest = lane_max(s_cur[0]);
      moved = __any(largest > kRescaleWatch);
      if (moved) raise(largest);
    }
    u32x4 pn[NKK];
    float rs = 0.f;
    const unsigned hwin = DROP ? dropout_window<BN / 2>(dkey, hrow + (unsigned)(t * (BN / 2)), hlow) : 0u;
    unsigned word_a = 0, word_b = 0;
    auto pair_of = [&](int e) DA_INLINE {      // registers 2 (e % 8) and the next of 32-key block e / 8
      const int kt = e / 8, r = 2 * (e % 8);
      h2 e2;
      e2[0] = (half_t)fast_exp2(s_cur[0][kt][r]);
      e2[1] = (half_t)fast_exp2(s_cur[0][kt][r + 1]);
      rs = add_pair(e2, rs);
      unsigned w2 = __builtin_bit_cast(unsigned, e2);
      if constexpr (DROP) {
        if (r % 4 == 0) dropout_bytes_shared(dropout_rounds(dkey, hwin + hstep[kt * 4 + r / 4]), dsel, word_a, word_b);
        w2 = dropout_clear_pair((r % 4 == 0) ? word_a : word_b, p.drop.threshold, w2);
      }
      pn[kt * 2 + r / 8][(r % 8) / 2] = w2;
    };
    constexpr int NV = kOpening ? 0 : NPV, NM = NV + NSC;     // matrix products of an iteration
    each<NM>([&](auto c_tag) DA_INLINE {
      // products alternate NV : NSC
      constexpr int c = decltype(c_tag)::value, npv = c * NV / NM, nsc = c - npv;
      if constexpr ((c + 1) * NV / NM > npv) {
        if constexpr (npv + VA < NPV) vfr[npv + VA] = vt_frag_at(npv + VA, VOFF);
        o[0][npv % NOT] = mfma32(vfr[npv], __builtin_bit_cast(h8, pw[npv / NOT]), o[0][npv % NOT]);
      } else {
        if constexpr (nsc + KA < NSC) ka[nsc + KA] = k_frag_at(nsc + KA, KOFF);
        constexpr int kt = nsc / NKS, ks = nsc % NKS;
        if constexpr (ks == 0) s_nxt[0][kt] = negm[0];
        s_nxt[0][kt] = mfma32(ka[nsc], qf[0][ks], s_nxt[0][kt]);
      }
      if constexpr (c == NM / 4) load_k2(tk, KP, tail);
      if constexpr (!kOpening && c == NM / 2) load_va(tv, VP, tail);
      if constexpr (!kOpening && c == 3 * NM / 4) load_vb(tv, VP, tail);
#pragma unroll
      for (int e = c * (8 * NKT) / NM; e < (c + 1) * (8 * NKT) / NM; ++e) pair_of(e);
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (!(POS & 1)) request_first(((POS + 2) % 4) * C::KBUF_BYTES, POS * C::VBUF_BYTES);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kWatching) {
      if (moved) lower();
    } else if (__builtin_expect(__any(rs > kRescaleSum), 0)) {
      ++moves;
      raise(lane_max(s_cur[0]));
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) s_nxt[0][kt][r] -= d;
      lower();
      rs = 0.f;
#pragma unroll
      for (int e = 0; e < 8 * NKT; ++e) pair_of(e);
    }
    l[0] += rs;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) pw[kk] = pn[kk];
    if constexpr (POS & 1) {
      wait_async_tiles();
      __syncthreads();
      request_first(((POS + 2) % 4) * C::KBUF_BYTES, POS * C::VBUF_BYTES);
    }
  };
  static_assert(!kLate || (C::PAIR && QS == 1), "a meeting every second tile");

  // One iteration: softmax of tile t (scores in s_cur) and its P*V product, overlapped with the score
  // product of tile t+1 (into s_nxt).
  // POS = (t + b0) % NBUF is the ring position: K tile t+1 is read from buffer POS+1 and V tile t from
  // buffer POS; K tile t+3 goes to buffer POS+3 (tile t-1, consumed two iterations ago) and V tile t+2 to
  // buffer POS+2 (tile t-2, likewise), all modulo NBUF.
  // `tail`: the iteration can meet tiles that reach past the last real key (their copies are clamped and, in
  // the padded variant, their keys masked); iterations that cannot are compiled without those tests.
  auto iteration = [&](int t, auto pos_tag, auto tail, f16v (&s_cur)[QS][NKT], f16v (&s_nxt)[QS][NKT]) DA_INLINE {
    constexpr int POS = decltype(pos_tag)::value;
    constexpr int KR = (POS + 1) % 4, KP = (POS + 3) % 4, VR = POS, VP = (POS + 2) % 4;
    // Asynchronous prefetch straight into LDS, two iterations ahead: K tile t+3 and V tile t+2.
    // The groups of load instructions are spread over the iteration so that the waves do not
    // queue up behind each other at the memory pipeline.
    const int tk = clampt(t + 3);
    const int tv = clampt(t + 2);
    constexpr bool kTail = TAIL && decltype(tail)::value, kLeanTail = kLean && kTail;
    load_k1(tk, KP, tail);

    static_assert(!(TAIL || DROP) || QS == 1, "one 32-row block per wave");
    if constexpr (kLeanTail) {
      // Before anything else of the iteration is requested, with no branch around it, from a lane number formed
      // anew, and with all of the iteration's copies, whose clamping takes registers too, in front of it: at D = 128
      // the loop fills the 256 registers, and kept apart like this the tail fits them as well (with branches, and
      // the copies spread as below, 260 bytes a lane went to scratch).
      load_k2(tk, KP, tail); load_va(tv, VP, tail); load_vb(tv, VP, tail);
      __builtin_amdgcn_sched_barrier(0);
      const int ln = lane_again();
      mask_scores(s_cur, (CAUSAL ? qt * BM + qw * 32 + (ln & 31) : p.n_keys - 1) - t * BN - 4 * (ln >> 5));
      __builtin_amdgcn_sched_barrier(0);
    }

    // K fragments of the next tile are requested first; the row maxima of this tile are reduced
    // while they arrive.
    h8 ka[NKT][NKS];
    read_k(KR * C::KBUF_BYTES, ka);

    if constexpr (kTail && !kLean) {
      // only the last tiles of a wave's loop reach past its first row, or hold padding keys
      if ((t + 1) * BN > (CAUSAL ? qt * BM + qw * 32 + 1 : p.n_keys))
        mask_scores(s_cur, (CAUSAL ? qt * BM + qw * 32 + j : p.n_keys - 1) - t * BN - 4 * g);
    }

    // The score product of the next tile goes to the matrix unit first and runs under the row maxima and
    // the exponentials of this tile.  It starts from the running reference as it stands before this
    // tile's update; when the update moves the reference, the few results are corrected with it.
    if constexpr (!kLeanTail) load_k2(tk, KP, tail);
    scores_of(ka, s_nxt, sc_first, sc_split);

    float mx[QS];
#pragma unroll
    for (int qs = 0; qs < QS; ++qs) mx[qs] = lane_max(s_cur[qs]);
    float mxall = mx[0];
#pragma unroll
    for (int qs = 1; qs < QS; ++qs) mxall = fmaxf(mxall, mx[qs]);
    // The reference only moves when some row of the wave outgrew it by more than the threshold
    // (always on the first tile, where it starts at 0 with nothing accumulated yet).
    if (__any(mxall > kRescaleThreshold) || t == 0) {
#pragma unroll
      for (int qs = 0; qs < QS; ++qs) {
        const float pm = pair_max(mx[qs]);
        const float d = (t == 0) ? pm : fmaxf(pm, 0.f);
        const float alpha = fast_exp2(-d);
        m[qs] += d;
        l[qs] *= alpha;
#pragma unroll
        for (int tt = 0; tt < NOT; ++tt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[qs][tt][r] *= alpha;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            s_cur[qs][kt][r] -= d;
            if (kt < KT_EARLY) s_nxt[qs][kt][r] -= d;     // the later ones start from the new reference
          }
#pragma unroll
        for (int r = 0; r < 16; ++r) negm[qs][r] = -m[qs];
        asm volatile("" : "+v"(negm[qs]));
      }
    }

    // From here on one basic block: the P*V product of this tile runs on the matrix unit while the
    // exponentials run on the VALU.
    // dropout: the mask arithmetic needs the registers of the K fragments, so the score product is
    // issued in full before the exponentials instead of between them
    if constexpr (DROP) __builtin_amdgcn_sched_barrier(0);

    // V^T fragments are requested PD products ahead of the product that uses them (measured: 2 and
    // 3 are 1.3 % faster than the single product the compiler picks by itself, 5 and 7 are not); the
    // first ones here, so that they arrive under the exponentials
    constexpr int PD = DROP ? 1 : 3;           // dropout: registers are short
    auto vt_frag = [&](int i) {
      const int kk = i / NOT, tt = i % NOT;
      const int off = VR * C::VBUF_BYTES + 16 * kk * DV * 2;
      return join(lds_read_tr_at(vtr[tt][0], off), lds_read_tr_at(vtr[tt][1], off));
    };
    h8 vfr[NPV];
    if constexpr (!DROP) {
#pragma unroll
      for (int i = 0; i < PD && i < NPV; ++i) vfr[i] = vt_frag(i);
    }
    scores_of(ka, s_nxt, sc_split, sc_end);

    // P^T as B operands: pb[kk] covers keys 16kk..16kk+15 (accumulator order).  Built from the packed
    // pairs as 32-bit words, so that each pair is converted once, for the row sum and the operand alike.
    u32x4 pw[QS][NKK];
#pragma unroll
    for (int qs = 0; qs < QS; ++qs) {
      float rs = 0.f;
      unsigned word_a = 0, word_b = 0;     // dropout: this query's bytes of the words of two neighbouring 2x2 blocks
      const unsigned hwin = DROP ? dropout_window<BN / 2>(dkey, hrow + (unsigned)(t * (BN / 2)), hlow) : 0u;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          h2 e2;
          e2[0] = (half_t)fast_exp2(s_cur[qs][kt][r]);
          e2[1] = (half_t)fast_exp2(s_cur[qs][kt][r + 1]);
          rs = add_pair(e2, rs);   // row sum of the rounded probabilities
          unsigned w2 = __builtin_bit_cast(unsigned, e2);
          if constexpr (DROP) {
            // registers r, r+1 hold the keys key, key+1 (key even) of this lane's query; the blocks of registers
            // r..r+1 and r+2..r+3 (r a multiple of 4) are neighbours, hashed one by each lane of a query pair
            if (r % 4 == 0) dropout_bytes_shared(dropout_rounds(dkey, hwin + hstep[kt * 4 + r / 4]), dsel, word_a, word_b);
            w2 = dropout_clear_pair((r % 4 == 0) ? word_a : word_b, p.drop.threshold, w2);
          }
          pw[qs][kt * 2 + r / 8][(r % 8) / 2] = w2;
        }
      l[qs] += rs;
    }

    if constexpr (DROP) {
#pragma unroll
      for (int i = 0; i < PD && i < NPV; ++i) vfr[i] = vt_frag(i);
    }
#pragma unroll
    for (int i = 0; i < NPV; ++i) {
      const int kk = i / NOT, tt = i % NOT;
      if (!kLeanTail && i == 0) load_va(tv, VP, tail);
      if (!kLeanTail && i == NPV / 2) load_vb(tv, VP, tail);
      if (i + PD < NPV) vfr[i + PD] = vt_frag(i + PD);
#pragma unroll
      for (int qs = 0; qs < QS; ++qs) o[qs][tt] = mfma32(vfr[i], __builtin_bit_cast(h8, pw[qs][kk]), o[qs][tt]);
    }

    // the tiles needed next were requested one iteration ago: only this iteration's loads may remain
    if constexpr (C::PAIR) {
      // the ring of four lets the workgroup meet every second tile only: the copies for the next two tiles
      // (requested during the last two) have landed for everybody, and the last two buffers may be refilled
      if constexpr (POS & 1) { wait_async_tiles(); __syncthreads(); }
    } else {
      wait_async_tiles_except(loads_per_iter);
      __syncthreads();
    }
  };

  auto one = [&](int t, auto pos_tag, auto tail, auto kind, f16v (&s_cur)[QS][NKT], f16v (&s_nxt)[QS][NKT]) DA_INLINE {
    if constexpr (kLate) late_iteration(t, pos_tag, tail, kind, s_cur, s_nxt);
    else iteration(t, pos_tag, tail, s_cur, s_nxt);
  };
  constexpr std::integral_constant<int, kOpens> opens{};
  constexpr std::integral_constant<int, kFollows> follows{};
  constexpr std::integral_constant<int, kWatches> watches{};
  // the tile count is even (N is a multiple of 128, tiles are at most 64 keys)
  int t = 0;
  if (head_half) {
    one(0, std::integral_constant<int, 2>{}, with_tail, opens, s_a, s_b);
    one(1, std::integral_constant<int, 3>{}, with_tail, follows, s_b, s_a);
    t = 2;
  }
  auto turn = [&](int t, auto tail, auto kind) DA_INLINE {
    one(t, std::integral_constant<int, 0>{}, tail, kind, s_a, s_b);
    one(t + 1, std::integral_constant<int, 1>{}, tail, kind, s_b, s_a);
    one(t + 2, std::integral_constant<int, 2>{}, tail, kind, s_a, s_b);
    one(t + 3, std::integral_constant<int, 3>{}, tail, kind, s_b, s_a);
  };
  if constexpr (TAIL) {
    // A mask concerns the last tiles only: with padding, an iteration copies K tile t+3, so the first one that can
    // touch a tile with padding rows is number n_keys / BN - 3; under the causal mask the workgroup's rows see all
    // of the tiles in front of its own.  Whole turns in front of both run without the tests.
    int t_tail = CAUSAL ? qt * (BM / BN) : p.N / BN;
    if (p.n_keys < p.N) t_tail = min(t_tail, p.n_keys / BN - 3);
#pragma nounroll
    for (; t + 4 <= t_tail && !(kWatch && moves >= kWatchMoves); t += 4) { moves = 0; turn(t, no_tail, follows); }
  }
#pragma nounroll
  for (; t < n_tiles && !(kWatch && moves >= kWatchMoves); t += 4) { moves = 0; turn(t, with_tail, follows); }
  if constexpr (kWatch) {
    if (__builtin_expect(moves >= kWatchMoves, 0)) {
#pragma nounroll
      for (; t < n_tiles; t += 4) turn(t, with_tail, watches);
    }
  }

  if constexpr (kLate) {
    // the last tile's product
    constexpr int VOFF = 3 * C::VBUF_BYTES;
#pragma unroll
    for (int i = 0; i < NPV; ++i)
      o[0][i % NOT] = mfma32(i < VA ? vfirst[i] : vt_frag_at(i, VOFF), __builtin_bit_cast(h8, pw[i / NOT]), o[0][i % NOT]);
  }
  wait_async_tiles();   // the staging blocks below reuse the tile memory the last prefetches write to
  __syncthreads();
  // ---- epilogue ----------------------------------------------------------------------------
  // Every row quantity is per query = per lane pair (l, l^32).  Each wave has a staging block of
  // 32 rows x DV halfs in the now idle tile memory (row stride DV+8 halfs).  Results are written
  // there in accumulator layout (8 bytes per lane) and read back row by row, so that the global
  // stores are whole 16-byte chunks of consecutive rows.  The stream-2 waves stage softmax(S2)V
  // rounded to 16 bits -- the tensor saved for backward -- and also hand it, unrounded, to the stream-1
  // wave that owns the same rows: the lambda-combine is formed in fp32, as in the reference
  // (src/kernel.py:191-194), so that rows in which the two streams nearly cancel (lambda near 1, similar
  // attention maps) do not see the rounding error of one stream amplified by the norm.  The two waves
  // hold a row's values in the same lanes and registers, so the exchange is lane to lane.
  // Each pair of waves has one block of tile memory: first it carries the fp32 exchange, then, once the
  // workgroup has met behind the combine, the staged rows of the two waves side by side.
  const int lane_e = lane_again(), j_e = lane_e & 31, g_e = lane_e >> 5;
  constexpr int SROW = DV + 8;
  float* const xch = reinterpret_cast<float*>(smem + (size_t)qw * C::XCH_BLOCK);
  half_t* const stg_own = smem + (size_t)qw * C::XCH_BLOCK + (st ? 32 * SROW : 0);
  auto stage_rows = [&](int qs, const f16v (&val)[NOT], float scale) {
#pragma unroll
    for (int tt = 0; tt < NOT; ++tt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        h4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (half_t)(val[tt][4 * r4 + e] * scale);
        *reinterpret_cast<h4*>(stg_own + j_e * SROW + 32 * tt + 8 * r4 + 4 * g_e) = v;
      }
    (void)qs;
  };
  // `rows`: how many of the wave's 32 rows exist in the destination (32 unless the sequence is padded and
  // the destination is the caller's tensor, which has no rows past the real length)
  // `gain`: null, or the factors of the DV features (a lane stores the same eight of every row).  Stored from here the
  // product costs its bytes once; as a launch of its own it read y back: a layer's step B8 H8 N1024 D64 439 -> 430 us, its
  // inference 138 -> 134, B2 H8 N512 D32 68 -> 64.  The operator's own calls, which have no gain, pay two tests of a pointer for
  // it: 1423 us with and 1425 without them at B2 H32 N4096 D128 fp16, 246 and 247 at B4 H32 N2048 D64 bf16 causal.
  auto store_rows = [&](half_t* gbase /* first of this wave's 32 rows */, size_t row_stride, int rows, const half_t* gain) {
    constexpr int LPR = DV / 8;            // lanes per row
    constexpr int RPI = 64 / LPR;          // rows per instruction
    const int ch = lane_e % LPR;
    h8 gv = {};
    if (gain) gv = *reinterpret_cast<const h8*>(gain + 8 * ch);
#pragma unroll
    for (int k = 0; k < 32 / RPI; ++k) {
      const int row = k * RPI + lane_e / LPR;
      u32x4 v = *reinterpret_cast<const u32x4*>(stg_own + row * SROW + 8 * ch);
      if (gain) {
        h8 x = __builtin_bit_cast(h8, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (half_t)((float)x[e] * (float)gv[e]);
        v = __builtin_bit_cast(u32x4, x);
      }
      if (!TAIL || row < rows) *reinterpret_cast<u32x4*>(gbase + (size_t)row * row_stride + 8 * ch) = v;
    }
  };

  static_assert(QS == 1, "the epilogue stages one 32-row block per wave");
  const float lsum = pair_sum(l[0]);
  const float inv = (DROP ? p.drop.keep_scale : 1.0f) / lsum;
  const size_t row = (size_t)bh * p.N + qt * BM + qw * 32 + j_e;
  const size_t wave_row0 = (size_t)bh * p.N + qt * BM + qw * 32;
  {
    float* lse = st ? p.lse2 : p.lse1;
    if (g_e == 0 && lse) lse[row] = (m[0] + __builtin_log2f(lsum)) * kLn2;
  }
  if (st == 1) {
#pragma unroll
    for (int tt = 0; tt < NOT; ++tt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        f4v u;
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = o[0][tt][4 * r4 + e] * inv;
        *reinterpret_cast<f4v*>(xch + ((tt * 4 + r4) * 64 + lane_e) * 4) = u;
      }
  }
  __syncthreads();
  float ss = 0.f;
  if (st == 0) {
#pragma unroll
    for (int tt = 0; tt < NOT; ++tt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f4v u = *reinterpret_cast<const f4v*>(xch + ((tt * 4 + r4) * 64 + lane_e) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = o[0][tt][4 * r4 + e] * inv - lam * u[e];
          o[0][tt][4 * r4 + e] = x;
          ss += x * x;
        }
      }
  }
  __syncthreads();      // the exchange has been read: the blocks may take the staged rows
  if (st == 1) {
    stage_rows(0, o[0], inv);
    __builtin_amdgcn_wave_barrier();   // the rows are read back by other lanes of this wave only
    if (p.u2) store_rows(p.u2 + wave_row0 * DV, DV, 32, nullptr);
  } else {
    float scale = 1.0f;
    if (RMS) {
      ss = pair_sum(ss);
      const float rr = __builtin_amdgcn_rsqf(ss * (1.0f / DV) + kEps);
      scale = (1.0f - p.lambda_init) * rr;
      if (g_e == 0 && p.rinv) p.rinv[row] = rr;
    }
    stage_rows(0, o[0], scale);
    __builtin_amdgcn_wave_barrier();   // the rows are read back by other lanes of this wave only
    const size_t out0 = da_abi::unit_base(p, p.sy, bh) + (size_t)(qt * BM + qw * 32) * (size_t)p.sy.n;
    const int out_rows = p.n_keys - (qt * BM + qw * 32);
    if (p.y) store_rows(p.y + out0, (size_t)p.sy.n, out_rows, nullptr);
    if (p.y_gain) store_rows(p.y_gain + out0, (size_t)p.sy.n, out_rows, p.gain);
  }
}

template <int D, bool RMS, bool DROP, bool SMALL>
static void launch_fwd_c(const FwdParams& p, hipStream_t stream) {
  using C = FwdCfg<D, SMALL>;
  const dim3 grid(p.BH * (p.N / C::BM)), block(C::NT);
  if (p.causal)
    hipLaunchKernelGGL((fwd_kernel<D, RMS, 1, DROP, SMALL>), grid, block, 0, stream, p);
  else if (p.n_keys < p.N)
    hipLaunchKernelGGL((fwd_kernel<D, RMS, 2, DROP, SMALL>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((fwd_kernel<D, RMS, 0, DROP, SMALL>), grid, block, 0, stream, p);
}

template <int D>
static hipError_t launch_fwd_t(const FwdParams& p, hipStream_t stream) {
  const bool drop = p.drop.threshold != 0;
  // The D = 128 dropout instantiations do not fit the 256 registers of the 128-row workgroup (two waves per SIMD) and
  // always run in 64-row workgroups at one wave per SIMD.
  const bool small_grid = da_abi::fwd_64_rows(D, p.causal, p.N, (long long)p.BH * (p.N / 128));
  if constexpr (D == 128) {
    if (drop) {
      if (p.rms_norm) launch_fwd_c<D, true, true, true>(p, stream); else launch_fwd_c<D, false, true, true>(p, stream);
    } else if (small_grid) {
      if (p.rms_norm) launch_fwd_c<D, true, false, true>(p, stream); else launch_fwd_c<D, false, false, true>(p, stream);
    } else {
      if (p.rms_norm) launch_fwd_c<D, true, false, false>(p, stream); else launch_fwd_c<D, false, false, false>(p, stream);
    }
    return hipGetLastError();
  } else {
    auto launch = [&](auto drop_tag, auto small_tag) {
      constexpr bool DR = decltype(drop_tag)::value, SM = decltype(small_tag)::value;
      if (p.rms_norm) launch_fwd_c<D, true, DR, SM>(p, stream); else launch_fwd_c<D, false, DR, SM>(p, stream);
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if (small_grid) { if (drop) launch(yes, yes); else launch(no, yes); }
    else            { if (drop) launch(yes, no); else launch(no, no); }
    return hipGetLastError();
  }
}

// Tile-size choice per head dimension (replaces the reference's run-time autotuner,
// src/kernel.py:12-19): 128 query rows per workgroup; 64 keys per step for D <= 64, 32 for D = 128.
hipError_t launch_fwd(const FwdParams& p, int D, hipStream_t stream) {
  switch (D) {
    case 32:  return launch_fwd_t<32>(p, stream);
    case 64:  return launch_fwd_t<64>(p, stream);
    case 128: return launch_fwd_t<128>(p, stream);
    default:  return hipErrorInvalidValue;
  }
}

}  // namespace DA_NS
