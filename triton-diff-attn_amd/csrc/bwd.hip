// Differential-attention backward for gfx950.  Same mathematics as the reference's fused backward
// (src/kernel.py:221-458) but split into stream-ordered kernels, which removes the reference's
// in-launch dependency between the row preprocess and the main loops:
//
//   bwd_prep_kernel   per row: RMSNorm backward (src/kernel.py:283-290), the two row dots
//                     delta1/delta2 (:295-296), d(lambda) partials (:293); writes dX in fp16 and
//                     the four row statistics the main kernels need.
//   bwd_dkdv_kernel   one workgroup per 128 keys, loops over all query tiles:
//                     dV += (P1 - lambda P2)^T dX, dK_t += s dS_t^T Q_t      (:410-424)
//   bwd_dq_kernel     one workgroup per 256 or 128 queries, loops over all key tiles:
//                     dQ_t += s dS_t K_t                                      (:426-436)
//   bwd_pair_kernel   blocks of both kinds in one grid: always at D = 128 without dropout, else where
//                     bwd_one_grid (dispatch.hpp) says so
//   d(lambda)         fixed-order sum of the partials into one fp16 value (one per head with per-head
//                     lambda) (:573): one extra workgroup per value at the end of the first grid of dK/dV or dQ
//                     blocks of the call, or bwd_dlambda_kernel when there is none
//
// The pre-norm row X is rebuilt as Y / ((1 - lambda_init) * rinv); only U2 = softmax(S2) V is
// needed besides it, because U1 = X + lambda U2.
#include <type_traits>

#include "dispatch.hpp"
#include "params.hpp"

namespace DA_NS {

constexpr int kPrepRows = 64;   // rows per workgroup of the preprocess kernel = one d(lambda) partial

int bwd_num_partials(int BH, int N, int D) { (void)D; return (int)(((long long)BH * N) / kPrepRows); }

// ------------------------------------------------------------------------------------------------
// GAIN: the caller's output was y times a gain per feature, and dy is the gradient of that product: it is multiplied by the
// gain on the way in, rounded to 16 bits as the product of two tensors is (d(lambda) is a sum of both signs that leaves little
// of them, and shows in its third digit whether that rounding was done), and the workgroup leaves the sum of dy * y over its rows, one value per
// feature, as its partial of the gain's gradient.  (As passes of their own, B8 H8 N1024 D64: 39 us for the two products and
// the sum, beside 15 us for this kernel.)
template <int D, bool RMS, bool GAIN = false>
__global__ __launch_bounds__(256) void bwd_prep_kernel(BwdParams p) {
  constexpr int DV = 2 * D, LPR = DV / 8, RPP = 256 / LPR;
  static_assert(RMS || !GAIN, "a gain multiplies normalised heads");
  __shared__ float red[GAIN ? RPP * DV : 256];
  const int tid = threadIdx.x, sub = tid % LPR, rloc = tid / LPR;
  // the 64 rows of a workgroup belong to one (batch, head) unit: N is a multiple of 128
  const int bh = (int)(((size_t)blockIdx.x * kPrepRows) / p.N);
  const int n0 = (int)(((size_t)blockIdx.x * kPrepRows) % p.N);
  const float lam = da_abi::lambda_of_unit(p, bh);
  const half_t* gy = p.y + da_abi::unit_base(p, p.sy, bh) + 8 * sub;
  const half_t* gdy = p.dy + da_abi::unit_base(p, p.sdy, bh) + 8 * sub;
  const float c = 1.0f - p.lambda_init;
  const size_t rows = (size_t)p.BH * p.N;
  // With dropout every probability of the other two kernels carries the factor c of the kept pairs (its logarithm is in
  // statistics 0 and 1), and the row dots carry 1/c; without, the factor is 1 and nothing changes.
  const bool drop = p.drop.threshold != 0;
  const float drop_inv = (float)(256u - p.drop.threshold) * (1.0f / 256.0f), drop_log2 = drop ? -log2f(drop_inv) : 0.f;
  float part = 0.f;
  float gain[8], gpart[8];
  if constexpr (GAIN) {
    const h8 v = *reinterpret_cast<const h8*>(p.gain + 8 * sub);
#pragma unroll
    for (int e = 0; e < 8; ++e) { gain[e] = (float)v[e]; gpart[e] = 0.f; }
  }
#pragma unroll 1
  for (int pass = 0; pass < kPrepRows / RPP; ++pass) {
    const size_t row = (size_t)blockIdx.x * kPrepRows + pass * RPP + rloc;
    const size_t off = row * DV + 8 * sub;
    const size_t n = (size_t)(n0 + pass * RPP + rloc);
    // a padding row (past the sequence's real length) has no y and dy rows: it gets dX = 0 and zero statistics,
    // so it adds nothing to dK, dV and d(lambda)
    const bool real = n < (size_t)p.n_keys;
    h8 y8, g8;
#pragma unroll
    for (int e = 0; e < 8; ++e) { y8[e] = (half_t)0.f; g8[e] = (half_t)0.f; }
    if (real) {
      y8 = *reinterpret_cast<const h8*>(gy + n * (size_t)p.sy.n);
      g8 = *reinterpret_cast<const h8*>(gdy + n * (size_t)p.sdy.n);
    }
    const h8 u8 = *reinterpret_cast<const h8*>(p.u2 + off);
    if constexpr (GAIN) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { gpart[e] += (float)g8[e] * (float)y8[e]; g8[e] = (half_t)((float)g8[e] * gain[e]); }
    }
    // dX of the row, and ix with X = ix * Y (the pre-norm row rebuilt from the saved output)
    float dx[8], ix = 1.0f;
    if (RMS) {
      float gy = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) gy = dot_pair(h2{g8[e], g8[e + 1]}, h2{y8[e], y8[e + 1]}, gy);
#pragma unroll
      for (int msk = LPR / 2; msk >= 1; msk >>= 1) gy += __shfl_xor(gy, msk, 64);
      const float r = p.rinv[row];
      if (c != 0.f) {
        const float a = c * r, b = r * gy / (c * DV);
        ix = 1.0f / (c * r);
#pragma unroll
        for (int e = 0; e < 8; ++e) dx[e] = a * (float)g8[e] - b * (float)y8[e];
      } else {
        ix = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) dx[e] = 0.f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) dx[e] = (float)g8[e];
    }
    // The row sums are formed from dX as the other kernels will read it, rounded to 16 bits: dS = A (dP - delta)
    // with dP = dX V^T cancels almost completely where a row attends to a single key, and a delta from the
    // unrounded dX would leave the rounding error of dX times V behind, scaled by a norm factor that is large
    // exactly in the rows where the two streams nearly cancel.  (The reference takes delta from the unrounded
    // gradient, src/kernel.py:290-296, and dP from the rounded one, :374-375 and :419.)  The products of the
    // 16-bit values are exact and summed in fp32.
    float t2 = 0.f, ty = 0.f;
    h8 d8;
#pragma unroll
    for (int e = 0; e < 8; ++e) d8[e] = (half_t)dx[e];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      t2 = dot_pair(h2{d8[e], d8[e + 1]}, h2{u8[e], u8[e + 1]}, t2);
      ty = dot_pair(h2{d8[e], d8[e + 1]}, h2{y8[e], y8[e + 1]}, ty);
    }
#pragma unroll
    for (int msk = LPR / 2; msk >= 1; msk >>= 1) {
      t2 += __shfl_xor(t2, msk, 64);
      ty += __shfl_xor(ty, msk, 64);
    }
    const float tx = ty * ix;      // rowsum(dX * X)
    *reinterpret_cast<h8*>(p.dx + off) = d8;
    if (sub == 0) {
      const float delta2 = -lam * t2;
      p.stat[0 * rows + row] = drop_log2 - p.lse1[row] * kLog2e;
      p.stat[1 * rows + row] = drop_log2 - p.lse2[row] * kLog2e;
      const float delta1 = tx - delta2;
      p.stat[2 * rows + row] = -delta1 * drop_inv;
      p.stat[3 * rows + row] = drop ? -delta2 * drop_inv : -(lam * delta1 + delta2);
      part -= t2;
    }
  }
  red[tid] = part;
  __syncthreads();
#pragma unroll
  for (int s = 128; s >= 1; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) p.dlam_part[blockIdx.x] = red[0];
  if constexpr (GAIN) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) red[rloc * DV + 8 * sub + e] = gpart[e];
    __syncthreads();
    for (int f = tid; f < DV; f += 256) {
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < RPP; ++r) sum += red[r * DV + f];
      p.dgain_part[(size_t)blockIdx.x * DV + f] = sum;
    }
  }
}

// Output o of n_out is the sum of the partials of the units o, o + n_out, o + 2 n_out, ...: with n_out = 1
// every unit (one lambda), with n_out = H the units of head o (one lambda per head).  `per_unit`
// consecutive partials belong to a unit.  One workgroup per output.  The sum is formed over 256 slots and a
// binary tree in a fixed order; a workgroup of fewer threads lets each thread play several slots, so the
// result does not depend on the kernel that hosts the reduction.
__device__ __forceinline__ void dlambda_reduce(const float* __restrict__ part, int per_unit, int n_units, half_t* out,
                                               int o, int n_out, float* red, int out_fp32) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int n = (n_units / n_out) * per_unit;        // partials this workgroup sums
  for (int slot = tid; slot < 256; slot += nt) {
    float acc = 0.f;
    if (n_out == 1) {
      for (int i = slot; i < n; i += 256) acc += part[i];
    } else {
      for (int i = slot; i < n; i += 256) acc += part[(size_t)(o + (i / per_unit) * n_out) * per_unit + i % per_unit];
    }
    red[slot] = acc;
  }
  __syncthreads();
#pragma unroll
  for (int s = 128; s >= 1; s >>= 1) {
    for (int slot = tid; slot < s; slot += nt) red[slot] += red[slot + s];
    __syncthreads();
  }
  if (tid == 0) {
    // the sum leaves the library in the 16-bit type of the tensors, like the reference's (src/kernel.py:573),
    // or unrounded in fp32 when the caller keeps lambda in fp32
    if (out_fp32) reinterpret_cast<float*>(out)[o] = red[0];
    else out[o] = (half_t)red[0];
  }
}

__global__ __launch_bounds__(256) void bwd_dlambda_kernel(const float* __restrict__ part, int per_unit, int n_units,
                                                          half_t* out, int out_fp32) {
  __shared__ float red[256];
  dlambda_reduce(part, per_unit, n_units, out, blockIdx.x, gridDim.x, red, out_fp32);
}

// The dK/dV and dQ kernels can host that reduction in p.dlam_fold extra workgroups at the end of their grid
// (one launch less per backward): such a workgroup does nothing else.
#define DA_HOST_DLAMBDA(smem_)                                                                                  \
  if (p.dlam_fold && (int)blockIdx.x >= (int)gridDim.x - p.dlam_fold) {                                         \
    dlambda_reduce(p.dlam_part, p.n_part / p.BH, p.BH, p.dlambda, (int)blockIdx.x - ((int)gridDim.x - p.dlam_fold), \
                   p.dlam_fold, reinterpret_cast<float*>(smem_), p.lambda_fp32);                                \
    return;                                                                                                     \
  }

// ------------------------------------------------------------------------------------------------
template <int D, bool CAUSAL>
struct DkvCfg {
  static constexpr int DV = 2 * D;
  static constexpr int NW = 4;                 // waves per workgroup, 32 keys each
  static constexpr int NT = NW * 64;
  static constexpr int BK = NW * 32;           // keys per workgroup
  // Query rows per staged tile.  The workgroup meets once per tile: with 32 rows at D = 64 twice as often, which costs 1.6 % (671 ->
  // 682 us at B4 H32 N2048).  Causal blocks take it all the same: with 64 rows a loop may begin in three ways (an odd half turn of
  // the ring, masked or not), and at the place where they join 110 to 300 bytes a lane went to scratch; with 32 a turn of the ring is
  // four sub-tiles, as is the diagonal block.
  static constexpr int BQ = (D <= 64 && !CAUSAL) ? 64 : 32;
  static constexpr int Q_TILE = BQ * D;        // halfs (swizzled, unpadded)
  static constexpr int X_TILE = BQ * DV;
  static constexpr int STAT = 4 * BQ * 2;      // 4 float arrays, counted in halfs
  static constexpr int STAGE = 2 * Q_TILE + X_TILE + STAT;
  // LDS map in bytes: the ring buffers of each kind of tile are contiguous, so that any buffer of a kind
  // is within the 64 KiB reach of an LDS instruction's immediate offset from one per-lane address
  static constexpr int QBUF = 2 * Q_TILE * 2, XBUF = X_TILE * 2, SBUF = STAT * 2;   // one ring buffer of Q1|Q2, dX, statistics
  // A staged tile is read from half a step before its first sub-tile is scored until half a step after its last one was,
  // while another is being fetched.  With one sub-tile per tile that takes the ring's four buffers: behind its meeting, step i reads tiles i
  // and i+1 and the first fragments of i+2, and tile i+3 is on its way into the buffer of i-1.  With two sub-tiles per tile three would
  // do.  The position of every step is known at compile time (the loop is unrolled over one turn of the ring, and the number
  // of steps is a multiple of four): every LDS address is then a per-lane register plus an immediate offset, with no address
  // arithmetic inside the loop.
  static constexpr int NBUF = 4;
  static constexpr int XBASE = NBUF * QBUF, SBASE = XBASE + NBUF * XBUF;
  static_assert(NBUF * QBUF <= 65536 && NBUF * XBUF <= 65536, "immediate offsets reach every buffer");
  static constexpr int SMEM = NBUF * STAGE;
};

// dK_t and dV for one block of keys.  Products are formed as [queries x keys] so that a lane owns
// one key column; P and dS in accumulator layout are then directly the A operands (rows = keys,
// contraction over queries) of dV = P^T dX and dK_t = dS_t^T Q_t.
// MODE 0 computes dV, dK1 and dK2 in one pass.  At D = 128 their accumulators plus the resident
// K1, K2, V rows exceed the 512 registers of a lane, so there are two kinds of key blocks, side by side in
// bwd_pair_kernel's grid and with dropout in two launches: MODE 1 computes dV only (scores S1, S2; no dP),
// MODE 2 computes dK1 and dK2 only.
// CAUSAL: queries before the key block are skipped and the four sub-tiles on the diagonal are masked.
// DROP: dropout on both softmax maps, masks regenerated from the hash the forward used.  With the
// keep mask m_t and c = 1/(1-p):  dS1 = A1 (c m1 dP - delta1),  dS2 = A2 (-lambda c m2 dP - delta2),
// dV = c (m1 A1 - lambda m2 A2)^T dX; delta1, delta2 are the row dots with the dropped-out U1, U2.  The preprocess folds
// c into the statistics, so that P_t = c A_t comes out of the exponential and, with K_t = m_t P_t,
// dS1 = K1 dP - P1 delta1/c,  dS2 = -lambda K2 dP - P2 delta2/c,  dV = (K1 - lambda K2)^T dX.  398 vector instructions
// a 32-query step instead of 476 with c, two masks of dP and statistic 3 formed in the loop; B4 H32 N2048 D64 fp16 878 -> 869 us
// and dQ 567 -> 555: the wave issued 5 % shorter, and 3 of that came back as waits.  It issues for 67 % of its time, for 17 % a
// unit does not take its next instruction and for 16 % it waits for LDS data or a barrier.  (Masks by sign bits instead of
// compare and select, and the two streams' hashes in step, change nothing on top of it.)
// PADDED: rows n_keys..N-1 are padding.  As queries they read the last real row of Q1 and Q2 (the row the
// forward used for their logsumexp) and carry dX = 0; as keys they read the last real row of K1, K2, V and
// their results are not stored.
// The block is number `wg` of `n_wg`; smem: DkvCfg::SMEM halfs of tile memory.
template <int D, int MODE, bool CAUSAL, bool DROP, bool PADDED>
__device__ __forceinline__ void dkdv_block(const BwdParams& p, int wg, int n_wg, lds_half* smem) {
  using C = DkvCfg<D, CAUSAL>;
  constexpr int DV = C::DV, NW = C::NW, BK = C::BK, BQ = C::BQ;
  constexpr int NKS = D / 16, NKV = DV / 16, NDT = D / 32, NVT = DV / 32;
  constexpr bool DO_V = (MODE != 2), DO_K = (MODE != 1);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, g = lane >> 5;

  const int n_kt = p.N / BK;
  int bh, kt;
  if constexpr (CAUSAL) {   // the first key block of a unit is seen by the most queries
    const UnitBlock ub = longest_first(wg, p.BH);
    bh = ub.unit; kt = ub.rank;
  } else {
    const int tile = xcd_remap(wg, n_wg);
    bh = tile / n_kt; kt = tile % n_kt;
  }
  const size_t rows = (size_t)p.BH * p.N;
  const size_t row0 = (size_t)bh * p.N;
  const int key = kt * BK + wave * 32 + j;
  const int key_row = (PADDED && key >= p.n_keys) ? p.n_keys - 1 : key;    // the row this lane's key is read from
  // element offsets of the unit's first row and the row strides of the strided tensors
  const size_t qk_base = da_abi::unit_base(p, p.sqk, bh), v_base = da_abi::unit_base(p, p.sv, bh);
  const int qk_n = (int)p.sqk.n, v_n = (int)p.sv.n;

  const float c = p.sm_scale * kLog2e;
  const float lam = da_abi::lambda_of_unit(p, bh);
  // hash keys of this unit's two softmax streams (used with dropout only)
  const DropoutKey dkey1 = dropout_key(p.drop, 2u * bh), dkey2 = dropout_key(p.drop, 2u * bh + 1);
  const DropoutSel dsel = dropout_sel_key(key & 1);

  // persistent B operands: this lane's key row of K1, K2, V
  h8 kf1[NKS], kf2[NKS], vf[NKV];
  {
    const half_t* r1 = p.k1 + qk_base + (size_t)key_row * qk_n + 8 * g;
    const half_t* r2 = p.k2 + qk_base + (size_t)key_row * qk_n + 8 * g;
    const half_t* rv = p.v + v_base + (size_t)key_row * v_n + 8 * g;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      // pre-multiplied by sm_scale*log2(e): the score products come out in log2 units
      h8 x1 = *reinterpret_cast<const h8*>(r1 + 16 * ks);
      h8 x2 = *reinterpret_cast<const h8*>(r2 + 16 * ks);
#pragma unroll
      for (int e = 0; e < 8; ++e) { x1[e] = (half_t)((float)x1[e] * c); x2[e] = (half_t)((float)x2[e] * c); }
      kf1[ks] = x1; kf2[ks] = x2;
    }
    if constexpr (DO_K) {
#pragma unroll
      for (int kv = 0; kv < NKV; ++kv) vf[kv] = *reinterpret_cast<const h8*>(rv + 16 * kv);
    }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) { keep_in_agpr(kf1[ks]); keep_in_agpr(kf2[ks]); }
    if constexpr (DO_K) {
#pragma unroll
      for (int kv = 0; kv < NKV; ++kv) keep_in_agpr(vf[kv]);
    }
  }

  f16v dv[NVT], dk1[NDT], dk2[NDT];
#pragma unroll
  for (int t = 0; t < NVT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) dv[t][r] = 0.f;
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) { dk1[t][r] = 0.f; dk2[t][r] = 0.f; }

  using QTile = AsyncTile<BQ, D, NW>;
  using XTile = AsyncTile<BQ, DV, NW>;
  const half_t* gq1 = p.q1 + qk_base;
  const half_t* gq2 = p.q2 + qk_base;
  const half_t* gx = p.dx + row0 * DV;
  const unsigned q_off = QTile::lane_off(wave, lane, qk_n);
  // the 4 x BQ statistics of a query tile are one piece of 16*BQ bytes: lane l < BQ fetches
  // stat[l / (BQ/4)][4 * (l % (BQ/4)) .. +3]
  const float* gstat = p.stat + row0;
  const unsigned stat_off = (unsigned)(((size_t)(lane / (BQ / 4)) * rows + 4 * (lane % (BQ / 4))) * sizeof(float));
  constexpr int XH = (XTile::PER + 1) / 2;

  auto stage = [&](int qt, int buf, int part) DA_INLINE {
    lds_half* bq = smem + buf * (C::QBUF / 2);
    lds_half* bx = smem + (C::XBASE + buf * C::XBUF) / 2;
    // dX and the statistics come from the workspace, which has all N rows; Q1 and Q2 have n_keys.  With padding every copy of
    // theirs is clamped: a branch per copy cut the products of a step apart, and with the twice as many copies of 32-row tiles
    // causal blocks had become slower by it than they were with 64-row ones.  us of a whole backward, fp16, with 64-row tiles and
    // branches -> 32-row tiles and branches -> now: D32 H8 N130 causal 15.9 -> 16.7 -> 15.6, H4 N3000 76.5 -> 75.7 -> 72.7; D64 H4 N3000
    // causal 107.8 -> 111.0 -> 105.3; 64-row tiles as before: D32 H4 N3000 75.9 -> 72.2 -> 70.1, D64 107.8 -> 104.2 -> 101.0, H16 N77 18.7 -> 19.1 -> 18.1.
    if (part == 0) {
      if constexpr (PADDED) QTile::issue_clamped(gq1 + (size_t)qt * BQ * qk_n, bq, wave, lane, q_off, qk_n, p.n_keys - 1 - qt * BQ);
      else QTile::issue_at(gq1 + (size_t)qt * BQ * qk_n, bq, wave, lane, q_off, qk_n);
      if (wave == 0 && lane < BQ) async_copy16(reinterpret_cast<const half_t*>(gstat + (size_t)qt * BQ), stat_off, smem + (C::SBASE + buf * C::SBUF) / 2);
    } else if (part == 1) {
      if constexpr (PADDED) QTile::issue_clamped(gq2 + (size_t)qt * BQ * qk_n, bq + C::Q_TILE, wave, lane, q_off, qk_n, p.n_keys - 1 - qt * BQ);
      else QTile::issue_at(gq2 + (size_t)qt * BQ * qk_n, bq + C::Q_TILE, wave, lane, q_off, qk_n);
    } else if (part == 2) {
      XTile::template issue<0, XH>(gx + (size_t)qt * BQ * DV, bx, wave, lane);
    } else {
      XTile::template issue<XH, XTile::PER>(gx + (size_t)qt * BQ * DV, bx, wave, lane);
    }
  };

  const int tr_row = 4 * g + ((lane & 15) >> 2);  // transposing reads: row inside a 16-row k-step
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  // Per-lane LDS byte addresses, computed once.  The XOR swizzle makes the address of a fragment a
  // different function of the lane for every 16-byte chunk column, so there is one register per chunk
  // column a lane ever reads; everything else (ring buffer, Q1 or Q2, sub-tile, k-step of 16 rows) is a
  // multiple of 16 rows, which the swizzle does not see, and travels in the instruction's immediate offset.
  const unsigned lds0 = (unsigned)(unsigned long)smem;
  unsigned qb[NKS], xb[NKV], qtr[NDT][2], xtr[NVT][2], stb;
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) qb[ks] = lds0 + 2u * (unsigned)swz_off<D>(j, 16 * ks + 8 * g);
#pragma unroll
  for (int kv = 0; kv < NKV; ++kv) xb[kv] = lds0 + C::XBASE + 2u * (unsigned)swz_off<DV>(j, 16 * kv + 8 * g);
#pragma unroll
  for (int tt = 0; tt < NDT; ++tt)
#pragma unroll
    for (int e = 0; e < 2; ++e) qtr[tt][e] = lds0 + 2u * (unsigned)swz_off<D>(tr_row + 8 * e, 32 * tt + tr_col);
#pragma unroll
  for (int tt = 0; tt < NVT; ++tt)
#pragma unroll
    for (int e = 0; e < 2; ++e) xtr[tt][e] = lds0 + C::XBASE + 2u * (unsigned)swz_off<DV>(tr_row + 8 * e, 32 * tt + tr_col);
  stb = lds0 + C::SBASE + 16u * (unsigned)g;
  // kept as they are: the compiler neither folds constants into them nor recomputes them in the loop
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(qb[ks]));
#pragma unroll
  for (int kv = 0; kv < NKV; ++kv) asm volatile("" : "+v"(xb[kv]));
#pragma unroll
  for (int tt = 0; tt < NDT; ++tt) asm volatile("" : "+v"(qtr[tt][0]), "+v"(qtr[tt][1]));
#pragma unroll
  for (int tt = 0; tt < NVT; ++tt) asm volatile("" : "+v"(xtr[tt][0]), "+v"(xtr[tt][1]));
  asm volatile("" : "+v"(stb));
  auto lds_h8 = [](unsigned addr, int off) -> h8 { return lds_read_at<h8>(addr, off); };
  auto lds_tr = [](unsigned addr, int off) -> h4 { return lds_read_tr_at(addr, off); };

  // The loop runs over 32-query sub-tiles i (SPT per staged tile), software-pipelined inside the
  // wave.  Step i interleaves, instruction group by instruction group,
  //   the matrix products S1, S2, dP of sub-tile i+1          (matrix unit, A fragments from LDS)
  //   the element-wise work of sub-tile i, one register row at a time          (VALU)
  //   the products dV, dK1, dK2 over queries 16..31 of sub-tile i-1 during the first half of the
  //   step and over queries 0..15 of sub-tile i during the second half, as soon as the
  //   element-wise work has packed their operands              (matrix unit, B fragments from LDS)
  // The interleaving is written out in source order and pinned with scheduling barriers, because
  // the matrix products with AGPR-resident B fragments are opaque to the instruction scheduler.
  constexpr int SPT = BQ / 32;
  struct Scores { f16v s1, s2, dp; };
  struct Packed { h8 pc[2], d1[2], d2[2]; };   // A operands of the dV / dK1 / dK2 products
  constexpr int NPROD = 2 * NKS + (DO_K ? NKV : 0);   // score products per sub-tile (dP is needed for dK only)
  // the D = 128 instantiations with dropout are short of registers: they request one fragment ahead
  constexpr bool kShort = DROP && D == 128;
  // A fragments requested ahead of their product (measured in one GPU call: 4 is 1 % faster than 3 at D = 64 and
  // D = 128 and the same at D = 32; 5 and 6 spill in some instantiations and are not faster)
  constexpr int DEPTH = kShort ? 1 : 4;

  // Product k of a sub-tile: even k is k-step k/2 of dP, odd k alternates k-steps of S1 and S2, so
  // the three accumulation chains advance together; without dP (MODE 1) S1 and S2 alternate.
  static_assert(NKV == 2 * NKS, "every second product belongs to dP");
  auto prod_frag = [&](int buf, int qs, int k) -> h8 {
    if (!DO_K || (k & 1)) {
      const int t = DO_K ? (k >> 1) : k;
      return lds_h8(qb[t >> 1], buf * C::QBUF + (t & 1) * C::Q_TILE * 2 + qs * 32 * D * 2);
    }
    return lds_h8(xb[k >> 1], buf * C::XBUF + qs * 32 * DV * 2);
  };
  // The products read their resident operand from AGPRs through the inline-assembly form, for which the
  // compiler places no wait states: nothing may be spilled (a reloaded operand directly in front of such a
  // product would be read too early; the build checks that no backward kernel uses scratch memory) and no
  // VALU instruction may write an operand right in front of one (an assembly scan in the tests checks that).
  // The dropout instantiations, whose mask arithmetic makes the compiler shuffle operands, issue ordinary
  // (compiler-visible) matrix instructions instead: the compiler then places every wait state itself.
  auto prod_mfma = [&](int k, h8 a, Scores& out) DA_INLINE {
    if (!DO_K || (k & 1)) {
      const int t = DO_K ? (k >> 1) : k, ks = t >> 1;
      if (t & 1) out.s2 = DROP ? mfma32(a, kf2[ks], out.s2) : mfma32_bagpr(a, kf2[ks], out.s2);
      else       out.s1 = DROP ? mfma32(a, kf1[ks], out.s1) : mfma32_bagpr(a, kf1[ks], out.s1);
    } else {
      out.dp = DROP ? mfma32(a, vf[k >> 1], out.dp) : mfma32_bagpr(a, vf[k >> 1], out.dp);
    }
  };
  // Row statistics written by the preprocess kernel: 0: -lse1*log2e, 1: -lse2*log2e, 2: -delta1,
  // 3: -(lambda*delta1 + delta2); with dropout log2(c) is added to 0 and 1, and 2 and 3 are -delta1/c and -delta2/c.
  // Statistics 0..2 are the initial accumulator values of the three
  // product chains, so the matrix unit delivers s1 - lse1, s2 - lse2 (log2 units) and dP - delta1.
  auto stat4 = [&](int buf, int qs, int which, int r4) -> f4v {
    return lds_read_at<f4v>(stb, buf * C::SBUF + (which * BQ + qs * 32 + 8 * r4) * 4);
  };
  auto results_ready = [&](Scores& s) {
    if constexpr (DO_K) mfma_results_ready(s.s1, s.s2, s.dp);
    else mfma_results_ready(s.s1, s.s2);
  };
  // initial accumulator values of the rows 4*r4 .. 4*r4+3
  auto init_rows = [&](int buf, int qs, Scores& out, int r4) DA_INLINE {
    const f4v a = stat4(buf, qs, 0, r4), bq = stat4(buf, qs, 1, r4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { out.s1[4 * r4 + e] = a[e]; out.s2[4 * r4 + e] = bq[e]; }
    if constexpr (DO_K) {
      // with dropout the mask applies to dP alone, so -delta1 cannot ride in the accumulator
      const f4v cq = DROP ? f4v{0.f, 0.f, 0.f, 0.f} : stat4(buf, qs, 2, r4);
#pragma unroll
      for (int e = 0; e < 4; ++e) out.dp[4 * r4 + e] = cq[e];
    }
  };
  auto init_scores = [&](int buf, int qs, Scores& out) DA_INLINE {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) init_rows(buf, qs, out, r4);
  };
  // Element-wise work of accumulator register r (query row 8*(r/4) + 4g + (r%4)), split in three
  // stages that are issued one product apart, so that no VALU instruction waits on the one
  // before it: (1) exponentials, (2) products, (3) fp16 packing of a pair of rows.
  struct RowTmp { float p1[16], p2[16], u[16], ds1[16], ds2[16], pc[16], k1[16], k2[16]; unsigned w1, w2, w1b, w2b; };
  // `rel` (masked steps only) = key index minus the query index of register 0 of the sub-tile:
  // register r holds query 8*(r/4) + (r%4) relative to that, and a query before its key sees nothing
  auto ew1 = [&](int r, const f4v& st3, const f4v& st2, const Scores& in, RowTmp& t, auto masked_tag, int rel, int qbase) DA_INLINE {
    t.p1[r] = fast_exp2(in.s1[r]);
    t.p2[r] = fast_exp2(in.s2[r]);
    if constexpr (decltype(masked_tag)::value) {
      if (8 * (r / 4) + (r % 4) < rel) { t.p1[r] = 0.f; t.p2[r] = 0.f; }
    }
    if constexpr (DROP) {
      // register r holds query qbase + 8*(r/4) + (r%4) of this lane's key; registers r, r+1 (r even)
      // share the hash words of their 2x2 block, one word per softmax stream
      const unsigned query = (unsigned)(qbase + 8 * (r / 4) + (r % 4));
      // the blocks of registers r..r+1 and r+2..r+3 (r a multiple of 4) are neighbours, hashed one by each
      // lane of a key pair
      if ((r & 3) == 0) {
        const unsigned odd = (unsigned)key & 1u;
        dropout_bytes_shared(dropout_word(dkey1, (unsigned)p.N / 2, (query >> 1) + odd, (unsigned)key >> 1), dsel, t.w1, t.w1b);
        dropout_bytes_shared(dropout_word(dkey2, (unsigned)p.N / 2, (query >> 1) + odd, (unsigned)key >> 1), dsel, t.w2, t.w2b);
      }
      const bool keep1 = dropout_keep_half((r & 2) ? t.w1b : t.w1, r & 1, p.drop.threshold);
      const bool keep2 = dropout_keep_half((r & 2) ? t.w2b : t.w2, r & 1, p.drop.threshold);
      t.k1[r] = keep1 ? t.p1[r] : 0.f;
      t.k2[r] = keep2 ? t.p2[r] : 0.f;
      if constexpr (DO_K) {
        t.k2[r] *= -lam;
        t.p1[r] *= st2[r % 4];
        t.p2[r] *= st3[r % 4];
      }
      return;
    }
    if constexpr (DO_K) {
      t.u[r] = __builtin_fmaf(-lam, in.dp[r], st3[r % 4]);
      asm volatile("" : "+v"(t.p1[r]), "+v"(t.p2[r]), "+v"(t.u[r]));   // computed here, not moved to its use
    } else {
      asm volatile("" : "+v"(t.p1[r]), "+v"(t.p2[r]));
    }
  };
  auto ew2 = [&](int r, const Scores& in, RowTmp& t) DA_INLINE {
    if constexpr (DROP) {
      if constexpr (DO_K) {
        t.ds1[r] = __builtin_fmaf(t.k1[r], in.dp[r], t.p1[r]);
        t.ds2[r] = __builtin_fmaf(t.k2[r], in.dp[r], t.p2[r]);
        if constexpr (DO_V) t.pc[r] = t.k1[r] + t.k2[r];
      } else {
        t.pc[r] = __builtin_fmaf(-lam, t.k2[r], t.k1[r]);
      }
      return;
    }
    if constexpr (DO_K) {
      t.ds1[r] = t.p1[r] * in.dp[r];
      t.ds2[r] = t.p2[r] * t.u[r];
    }
    if constexpr (DO_V) t.pc[r] = __builtin_fmaf(-lam, t.p2[r], t.p1[r]);
    if constexpr (DO_K && DO_V) asm volatile("" : "+v"(t.ds1[r]), "+v"(t.ds2[r]), "+v"(t.pc[r]));
    else if constexpr (DO_K) asm volatile("" : "+v"(t.ds1[r]), "+v"(t.ds2[r]));
    else asm volatile("" : "+v"(t.pc[r]));
  };
  auto ew3 = [&](int r, const RowTmp& t, Packed& out) DA_INLINE {   // r odd: packs rows r-1 and r
    if constexpr (DO_V) { out.pc[r / 8][r % 8 - 1] = (half_t)t.pc[r - 1]; out.pc[r / 8][r % 8] = (half_t)t.pc[r]; }
    if constexpr (DO_K) {
      out.d1[r / 8][r % 8 - 1] = (half_t)t.ds1[r - 1]; out.d1[r / 8][r % 8] = (half_t)t.ds1[r];
      out.d2[r / 8][r % 8 - 1] = (half_t)t.ds2[r - 1]; out.d2[r / 8][r % 8] = (half_t)t.ds2[r];
    }
  };
  // slot s of the skewed schedule: stage 1 of row s, stage 2 of row s-1, stage 3 of the pair ending at row s-2
  auto ew_slot = [&](int s, const f4v (&st)[4], const f4v (&st2)[4], const Scores& in, RowTmp& t, Packed& out, auto masked_tag,
                     int rel, int qbase) DA_INLINE {
    if (s < 16) ew1(s, st[s / 4], st2[s / 4], in, t, masked_tag, rel, qbase);
    if (s >= 1 && s - 1 < 16) ew2(s - 1, in, t);
    if (s >= 2 && s - 2 < 16 && ((s - 2) & 1)) ew3(s - 2, t, out);
  };
  // B fragment (transposing read) of accumulate product m of sub-tile qs: m = kk*NACC1 + slot, where
  // the slots of a 16-query k-step are the dV feature tiles followed by the dK1/dK2 feature tiles
  constexpr int NSV = DO_V ? NVT : 0;          // dV slots
  constexpr int NACC1 = NSV + (DO_K ? 2 * NDT : 0);
  constexpr int NACC = 2 * NACC1;
  static_assert(NPROD % NACC == 0, "a whole number of score products per accumulate product");
  constexpr int RATIO = NPROD / NACC;
  auto acc_frag = [&](int buf, int qs, int m) -> h8 {
    const int kk = m / NACC1, slot = m % NACC1;
    const int row0 = qs * 32 + 16 * kk;
    if (slot < NSV) {
      const int off = buf * C::XBUF + row0 * DV * 2;
      return join(lds_tr(xtr[slot][0], off), lds_tr(xtr[slot][1], off));
    }
    const int t2 = slot - NSV;
    const int off = buf * C::QBUF + (t2 & 1) * C::Q_TILE * 2 + row0 * D * 2;
    return join(lds_tr(qtr[t2 >> 1][0], off), lds_tr(qtr[t2 >> 1][1], off));
  };
  auto acc_mfma = [&](int m, h8 bfrag, const Packed& in) DA_INLINE {
    const int kk = m / NACC1, slot = m % NACC1;
    if (slot < NSV) { dv[slot] = mfma32(in.pc[kk], bfrag, dv[slot]); return; }
    const int t2 = slot - NSV;
    if (t2 & 1) dk2[t2 >> 1] = mfma32(in.d2[kk], bfrag, dk2[t2 >> 1]);
    else        dk1[t2 >> 1] = mfma32(in.d1[kk], bfrag, dk1[t2 >> 1]);
  };

  const int n_qt = p.N / BQ;
  const int n_sub = p.N / 32;
  // first sub-tile and tile of the loop: with the causal mask no query before the key block matters
  const int i0 = CAUSAL ? kt * (BK / 32) : 0;
  const int t0 = i0 / SPT;
  // Tile t0 + k lives in buffer k % NBUF.  Step number s of the loop (sub-tile i0 + s) is at ring
  // position s % RING; the positions of its three sub-tiles follow from that at compile time.
  constexpr int NBUF = C::NBUF, RING = SPT * NBUF, HALF = RING / 2;
  static_assert(HALF % 2 == 0 && 4 % HALF == 0, "half a turn is an even number of steps and divides the step count");

  // One step.  Chunk k holds score product k of sub-tile i+1, every RATIO-th chunk also
  // accumulate product (k/RATIO + NACC/2) % NACC -- the upper query half of sub-tile i-1
  // during the first half of the step, then the lower query half of sub-tile i -- and
  // every chunk its share of the element-wise rows of sub-tile i.  `pk` holds the packed operands: its lower half is written
  // during the first half of the step and read during the second, its upper half is written during the second half and
  // read during the first half of the next step.
  // One wave per SIMD has nobody to hide the start of a step behind, so a step finds the first fragments of its products and
  // the initial values of its accumulators in registers: the step in front of it requested them, the initial values in the rows of
  // scores that it was done with.  For that the tile of sub-tile i+2 has to be there from the middle of step i on, where the workgroup
  // meets; it is requested behind the meeting of the step before (a tile of two sub-tiles: of two steps before).  When a step
  // requested all that at its own start, and the workgroup met there, behind copies requested as late as a quarter of a step before,
  // its products began 300 cycles late and a wave of the D = 128 kernel waited for 31 % of its time: us, key blocks alone, before ->
  // now, fp16: B2 H32 N4096 D128 3000 -> 2610, B4 H32 N2048 D64 687 -> 671, B2 H16 N8192 D32 1439 -> 1423 and, on another card,
  // 1365 -> 1388, which is even; with the query blocks in one grid B8 H32 N4096 D128 18.1 -> 16.7 ms, B1 H8 N2048 D64 79 -> 75 us, B2 H16
  // N512 D32 causal 18.1 -> 17.2.
  static_assert(NPROD % 16 == 0 || 16 % NPROD == 0, "rows are spread evenly over the products");
  constexpr int AHEAD = kShort ? 1 : 3;        // B fragments requested ahead of their product (4: no faster)
  // What a step finds requested by the step in front of it: the first fragments of its products and the statistics of its
  // first rows; its score accumulators hold their initial values.
  struct First { h8 a[DEPTH], b[AHEAD]; f4v st; };
  constexpr bool kCarry = !kShort;             // where registers are short a step requests its own
  First first;
  // the accumulate products of a step in their order: the upper query half of sub-tile (bufp, qsp), then the lower one of (bufc, qsc)
  auto step_bfrag = [&](int bufp, int qsp, int bufc, int qsc, int ja) -> h8 {
    const int m = (ja + NACC / 2) % NACC;
    return (ja < NACC / 2) ? acc_frag(bufp, qsp, m) : acc_frag(bufc, qsc, m);
  };
  auto request_first = [&](auto pos_tag) DA_INLINE {     // for the step at ring position POS
    constexpr int POS = decltype(pos_tag)::value;
    constexpr int SUBN = (POS + 1) % SPT, SUBC = POS % SPT, SUBP = (POS + RING - 1) % SPT;
    constexpr int BUFN = ((POS + 1) / SPT) % NBUF, BUFC = POS / SPT, BUFP = ((POS + RING - 1) / SPT) % NBUF;
#pragma unroll
    for (int k = 0; k < DEPTH; ++k) first.a[k] = prod_frag(BUFN, SUBN, k);
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) first.b[k] = step_bfrag(BUFP, SUBP, BUFC, SUBC, k);
    if constexpr (DO_K) first.st = stat4(BUFC, SUBC, 3, 0);
  };
  auto step = [&](int i, auto pos_tag, Scores& s_cur, Scores& s_nxt, Packed& pk, auto masked_tag) DA_INLINE {
    constexpr int POS = decltype(pos_tag)::value;
    // sub-tiles i-1 (p), i (c), i+1 (n) and i+2 (f)
    constexpr int SUBF = (POS + 2) % SPT, SUBN = (POS + 1) % SPT, SUBC = POS % SPT, SUBP = (POS + RING - 1) % SPT;
    constexpr int BUFF = ((POS + 2) / SPT) % NBUF, BUFN = ((POS + 1) / SPT) % NBUF, BUFC = POS / SPT, BUFP = ((POS + RING - 1) / SPT) % NBUF;
    constexpr bool meets = (SUBF == 0);
    const int rel = key - 32 * i - 4 * g, qbase = 32 * i + 4 * g;
    // Past the end the last tile is fetched and scored again and the result is never used.
    const int far = i / SPT + (SPT == 1 ? 3 : 2);
    const int tile_far = far < n_qt ? far : n_qt - 1;
    constexpr int BUF_FAR = (POS / SPT + (SPT == 1 ? 3 : 2)) % NBUF;
    constexpr int NSLOT = 18;                  // 16 rows + 2 slots of pipeline drain
    constexpr int LEAD = 2;                    // slots run before the first product
    // rows 0..7 are packed by slot 9, which must precede the first product that reads them
    static_assert(LEAD + (NSLOT - LEAD) * (NPROD / 2) / NPROD > 9, "lower half packed before it is read");
    h8 a[NPROD], bf[NACC];
    f4v st[4], st2[4];
    RowTmp tmp;
    if constexpr (!kCarry) {
      init_scores(BUFN, SUBN, s_nxt);
      request_first(pos_tag);
    }
#pragma unroll
    for (int k = 0; k < DEPTH; ++k) a[k] = first.a[k];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) bf[k] = first.b[k];
    st[0] = first.st;
    if constexpr (DO_K && DROP) {
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) st2[r4] = stat4(BUFC, SUBC, 2, r4);
    }
#pragma unroll
    for (int s = 0; s < LEAD; ++s) ew_slot(s, st, st2, s_cur, tmp, pk, masked_tag, rel, qbase);
    __builtin_amdgcn_sched_barrier(0);
    each<NPROD>([&](auto k_tag) DA_INLINE {
      constexpr int k = decltype(k_tag)::value;
      if constexpr (k == NPROD / 2 && meets) {
        // The tile of sub-tile i+2 has landed for everybody, and everybody is done with sub-tile i-1.
        wait_async_tiles();
        __syncthreads();
      }
      if constexpr (k + DEPTH < NPROD) a[k + DEPTH] = prod_frag(BUFN, SUBN, k + DEPTH);
      else if constexpr (kCarry) first.a[k + DEPTH - NPROD] = prod_frag(BUFF, SUBF, k + DEPTH - NPROD);
      if constexpr (k % RATIO == 0) {
        constexpr int ja = k / RATIO + AHEAD;
        if constexpr (ja < NACC) bf[ja] = step_bfrag(BUFP, SUBP, BUFC, SUBC, ja);
        else if constexpr (kCarry) first.b[ja - NACC] = step_bfrag(BUFC, SUBC, BUFN, SUBN, ja - NACC);
      }
      // statistics of the next row group, requested a quarter of a step ahead of their use
      if constexpr (DO_K && k % (NPROD / 4) == 0) {
        constexpr int r4 = k / (NPROD / 4) + 1;
        if constexpr (r4 < 4) st[r4] = stat4(BUFC, SUBC, 3, r4);
        else if constexpr (kCarry) first.st = stat4(BUFN, SUBN, 3, 0);
      }
      // the fetch of a tile is spread over the products so that the waves do not queue up at the memory pipeline
      if constexpr (SPT == 1) {
        if constexpr (k >= NPROD / 2 && (k - NPROD / 2) % (NPROD / 8) == 0) stage(tile_far, BUF_FAR, (k - NPROD / 2) / (NPROD / 8));
      } else {
        if constexpr (SUBC == 0 && k >= NPROD / 2 && k % (NPROD / 4) == 1) stage(tile_far, BUF_FAR, k / (NPROD / 4) - 2);
        if constexpr (SUBC == 1 && k < NPROD / 2 && k % (NPROD / 4) == 1) stage(tile_far, BUF_FAR, k / (NPROD / 4) + 2);
      }
      if constexpr (k % RATIO == 0) acc_mfma((k / RATIO + NACC / 2) % NACC, bf[k / RATIO], pk);
      prod_mfma(k, a[k], s_nxt);
      // slots LEAD .. NSLOT-1 spread over the products
      constexpr int s0 = LEAD + (NSLOT - LEAD) * k / NPROD, s1 = LEAD + (NSLOT - LEAD) * (k + 1) / NPROD;
#pragma unroll
      for (int s = s0; s < s1; ++s) ew_slot(s, st, st2, s_cur, tmp, pk, masked_tag, rel, qbase);
      // rows that are done with take the initial values of sub-tile i+2 (a row's last use is in the slot behind its own)
      if constexpr (kCarry && k >= NPROD / 2) {
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          if (s1 > 4 * r4 + 4 && !(s0 > 4 * r4 + 4 && k > NPROD / 2)) init_rows(BUFF, SUBF, s_cur, r4);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    // the next step's VALU reads these results right away
    results_ready(s_nxt);
  };

  // prologue: the last buffer, which the first step reads as "the sub-tile before the first", is cleared
  // (uninitialised LDS could hold NaN patterns, and 0 * NaN would poison the sums); the first tile is
  // fetched, then the second starts; scores of the first sub-tile
  const bool head_half = HALF == 4 && ((n_sub / HALF) & 1);
  const int b0 = head_half ? NBUF / 2 : 0;          // buffer of the first tile
  {
    const int bz = (b0 + NBUF - 1) % NBUF;          // the buffer in front of the first tile's
    DA_LDS u32x4* zq = (DA_LDS u32x4*)(smem + bz * (C::QBUF / 2));
    DA_LDS u32x4* zx = (DA_LDS u32x4*)(smem + (C::XBASE + bz * C::XBUF) / 2);
    for (int k = tid; k < C::QBUF / 16; k += C::NT) zq[k] = u32x4{0u, 0u, 0u, 0u};
    for (int k = tid; k < C::XBUF / 16; k += C::NT) zx[k] = u32x4{0u, 0u, 0u, 0u};
  }
  const int t1 = min(t0 + 1, n_qt - 1), t2 = min(t0 + 2, n_qt - 1);
  stage(t0, b0, 0); stage(t0, b0, 1); stage(t0, b0, 2); stage(t0, b0, 3);
  // the first step's second product reads the second tile where a tile is one sub-tile, else the tile in front of it
  if constexpr (SPT == 1) { stage(t1, b0 + 1, 0); stage(t1, b0 + 1, 1); stage(t1, b0 + 1, 2); stage(t1, b0 + 1, 3); }
  wait_async_tiles();
  __syncthreads();
  {
    constexpr int NEXT = SPT == 1 ? 2 : 1;
    const int tn = SPT == 1 ? t2 : t1, bn = (b0 + NEXT) % NBUF;
    stage(tn, bn, 0); stage(tn, bn, 1); stage(tn, bn, 2); stage(tn, bn, 3);
  }
  Scores sa, sb;
  Packed pk;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int e = 0; e < 8; ++e) { pk.pc[kk][e] = (half_t)0.f; pk.d1[kk][e] = (half_t)0.f; pk.d2[kk][e] = (half_t)0.f; }
  auto begin = [&](auto pos_tag) DA_INLINE {
    constexpr int POS = decltype(pos_tag)::value;
    init_scores(POS / SPT, 0, sa);
#pragma unroll
    for (int k = 0; k < NPROD; ++k) prod_mfma(k, prod_frag(POS / SPT, 0, k), sa);
    if constexpr (kCarry) {
      init_scores((POS + 1) / SPT, (POS + 1) % SPT, sb);
      request_first(pos_tag);
    }
  };
  if (head_half) begin(std::integral_constant<int, HALF>{});
  else begin(std::integral_constant<int, 0>{});
  results_ready(sa);

  // two steps, starting at the even ring position P0 with the scores of sub-tile i in sa
  auto two_steps = [&](int i, auto p0_tag, auto masked_tag) DA_INLINE {
    constexpr int P0 = decltype(p0_tag)::value;
    step(i, std::integral_constant<int, P0>{}, sa, sb, pk, masked_tag);
    step(i + 1, std::integral_constant<int, P0 + 1>{}, sb, sa, pk, masked_tag);
  };
  auto half_turn = [&](int i, auto h0_tag, auto masked_tag) DA_INLINE {
    constexpr int H0 = decltype(h0_tag)::value;
    two_steps(i, std::integral_constant<int, H0>{}, masked_tag);
    if constexpr (HALF == 4) two_steps(i + 2, std::integral_constant<int, H0 + 2>{}, masked_tag);
  };
  // The steps are a multiple of four.  Where a turn has eight the loop runs whole turns, and an odd half turn comes first,
  // at the ring's second half (the prologue has put the first tile into the buffer that goes with it).  With the causal mask
  // a turn has four: the key block's own four sub-tiles come first and straddle the diagonal, wave w masks sub-tiles i0 .. i0+w.
  static_assert(!CAUSAL || (BK == 128 && RING == 4), "four diagonal sub-tiles per key block, one turn of the ring");
  constexpr std::integral_constant<int, 0> first_half{};
  constexpr std::integral_constant<int, HALF> second_half{};
  int i = i0;
  if (head_half) {
    half_turn(i, second_half, std::false_type{});
    i += HALF;
  }
  if constexpr (CAUSAL) {
    half_turn(i, first_half, std::true_type{});
    half_turn(i + HALF, second_half, std::true_type{});
    i += RING;
  }
#pragma nounroll
  for (; i < n_sub; i += RING) {
    half_turn(i, first_half, std::false_type{});
    half_turn(i + HALF, second_half, std::false_type{});
  }
  // upper query half of the last sub-tile, at the last ring position
#pragma unroll
  for (int m = NACC / 2; m < NACC; ++m)
    acc_mfma(m, kCarry && m - NACC / 2 < AHEAD ? first.b[m - NACC / 2] : acc_frag((RING - 1) / SPT, (RING - 1) % SPT, m), pk);

  wait_async_tiles();   // the re-fetch issued by the last step has nothing left to land in after the kernel
  // accumulator tile tt: column = 32*tt + j (feature), register r = key row 8*(r/4) + 4g + (r%4)
  const int kloc0 = kt * BK + wave * 32;               // first key of this wave inside the unit
  if constexpr (DO_V) {
    half_t* const o = p.dv + da_abi::unit_base(p, p.sdv, bh) + (size_t)kloc0 * (size_t)p.sdv.n;
#pragma unroll
    for (int tt = 0; tt < NVT; ++tt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 8 * (r / 4) + 4 * g + (r % 4);
        if (!PADDED || kloc0 + kr < p.n_keys) o[(size_t)kr * (size_t)p.sdv.n + 32 * tt + j] = (half_t)dv[tt][r];
      }
  }
  if constexpr (DO_K) {
    const size_t ob = da_abi::unit_base(p, p.sdqk, bh) + (size_t)kloc0 * (size_t)p.sdqk.n;
#pragma unroll
    for (int tt = 0; tt < NDT; ++tt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 8 * (r / 4) + 4 * g + (r % 4);
        if (!PADDED || kloc0 + kr < p.n_keys) {
          p.dk1[ob + (size_t)kr * (size_t)p.sdqk.n + 32 * tt + j] = (half_t)(dk1[tt][r] * p.sm_scale);
          p.dk2[ob + (size_t)kr * (size_t)p.sdqk.n + 32 * tt + j] = (half_t)(dk2[tt][r] * p.sm_scale);
        }
      }
  }
}

template <int D, int MODE, bool CAUSAL, bool DROP, bool PADDED>
__global__ __launch_bounds__((DkvCfg<D, CAUSAL>::NT)) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_dkdv_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(16))) half_t smem[DkvCfg<D, CAUSAL>::SMEM];
  static_assert(sizeof(smem) >= 256 * sizeof(float), "the hosted reduction uses the tile memory");
  DA_HOST_DLAMBDA(smem)
  dkdv_block<D, MODE, CAUSAL, DROP, PADDED>(p, blockIdx.x, gridDim.x - p.dlam_fold, (lds_half*)smem);
}

// ------------------------------------------------------------------------------------------------
template <int D, int NWAVES, bool PIPE>
struct DqCfg {
  static constexpr int DV = 2 * D;
  static constexpr int NW = NWAVES;            // waves per workgroup, 32 query rows each
  // waves per SIMD the register budget is sized for: the resident Q1, Q2, dX rows and the two dQ
  // accumulators of a D = 128 wave do not fit 256 registers
  static constexpr int OCC = (D == 128 || PIPE) ? 1 : 2;
  static constexpr int NT = NW * 64;
  // thread count the register budget is derived from: with fewer than 4 * OCC waves in a workgroup
  // the occupancy attribute alone does not hold the allocator to 512 / OCC registers
  static constexpr int REG_NT = (OCC * 256 > NT) ? OCC * 256 : NT;
  static constexpr int BM = NW * 32;           // query rows per workgroup
  static constexpr int BN = (D <= 64) ? 64 : 32;  // keys per staged tile
  static constexpr int K_TILE = BN * D;        // halfs (swizzled, unpadded)
  static constexpr int V_TILE = BN * DV;
  static constexpr int STAGE = 2 * K_TILE + V_TILE;
  // A ring of four buffers whose position is a compile-time constant in every iteration (the loop body is one
  // turn of the ring), laid out by tile kind so that an instruction's immediate offset reaches every buffer.
  // Tiles are fetched two iterations ahead, in the pipelined form three, which takes the four buffers.  In the other form with a
  // barrier per tile three would do; four let the workgroup meet every second tile only (a tile's buffer is refilled two tiles
  // after it was read, which is always past one barrier), so the two waves of a SIMD, which leave a barrier in step, have twice
  // as long to drift apart and overlap one's matrix products with the other's element-wise work.  Measured in one GPU call
  // against a barrier per tile: 3.6 % faster at D = 128, 0.8 % at D = 32, 2 % slower at D = 64.
  static constexpr bool PAIR = (D != 64);      // a barrier every second tile
  static constexpr int NBUF = 4;
  static constexpr int KBUF_BYTES = 2 * K_TILE * 2, VBUF_BYTES = V_TILE * 2, VBASE_BYTES = NBUF * KBUF_BYTES;
  static_assert(NBUF * KBUF_BYTES <= 65536 && NBUF * VBUF_BYTES <= 65536, "immediate offsets reach every buffer");
  static constexpr int SMEM = NBUF * STAGE;
};

// dQ_t = s * dS_t K_t for one block of query rows.  Every product is formed transposed,
// [keys x queries], so that a lane owns one query column: the row statistics are per-lane
// scalars and dS^T in accumulator layout is directly the B operand of dQ^T = K^T dS^T.
// MASK: 0 none; 1 causal (key <= query); 2 the last keys of the sequence are padding (key < n_keys).
// A padded key has a zero K row, but its recomputed "probability" exp(0 - lse) is not small when a
// row's logsumexp is negative, and its dS can overflow fp16: it must be masked, not multiplied by 0.
// DROP: dropout on both softmax maps, as in bwd_dkdv_kernel.
// PIPE: one wave per SIMD, pipelined inside the wave.  The block is number `wg` of `n_wg`; smem: DqCfg::SMEM halfs.
template <int D, int NWAVES, int MASK, bool DROP, bool PIPE>
__device__ __forceinline__ void dq_block(const BwdParams& p, int wg, int n_wg, lds_half* smem) {
  using C = DqCfg<D, NWAVES, PIPE>;
  constexpr bool CAUSAL = (MASK == 1), PADDED = (MASK == 2);
  // rows past the real length are neither read from the caller's tensors nor written to the gradients: checked
  // in both masked variants (the causal one serves padded sequences too), compiled out of the plain one
  constexpr bool TAIL = (MASK != 0);
  constexpr int DV = C::DV, NW = C::NW, BM = C::BM, BN = C::BN;
  constexpr int NKS = D / 16, NKV = DV / 16, NDT = D / 32;
  constexpr bool kPipe = PIPE;     // the software-pipelined loop of the one-wave-per-SIMD kernel, below

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, g = lane >> 5;

  const int n_qt = p.N / BM;
  int bh, qt;
  if constexpr (CAUSAL) {   // the last query block of a unit sees the most keys
    const UnitBlock ub = longest_first(wg, p.BH);
    bh = ub.unit; qt = n_qt - 1 - ub.rank;
  } else {
    const int tile = xcd_remap(wg, n_wg);
    bh = tile / n_qt; qt = tile % n_qt;
  }
  const size_t rows = (size_t)p.BH * p.N;
  const size_t row0 = (size_t)bh * p.N;
  const size_t qrow = row0 + qt * BM + wave * 32 + j;
  // element offsets of the unit's first row and the row strides of the strided tensors
  const size_t qk_base = da_abi::unit_base(p, p.sqk, bh), v_base = da_abi::unit_base(p, p.sv, bh);
  const int qk_n = (int)p.sqk.n, v_n = (int)p.sv.n;

  const float lam = da_abi::lambda_of_unit(p, bh);
  // used with dropout only, as in the forward: hash keys of this unit's two softmax streams, the counter of this
  // query's first key pair, the counters' lane-dependent low bits, and what a block of eight keys adds
  const DropoutKey dkey1 = dropout_key(p.drop, 2u * bh), dkey2 = dropout_key(p.drop, 2u * bh + 1);
  const unsigned hquery = (unsigned)(qt * BM + wave * 32 + j);
  const unsigned hrow = (hquery >> 1) * ((unsigned)p.N / 2), hlow = 2u * (unsigned)g + (hquery & 1u);
  const DropoutSel dsel = dropout_sel_query(hquery & 1u);
  unsigned hstep1[4], hstep2[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) { hstep1[v] = dropout_window_step<16>(dkey1, v); hstep2[v] = dropout_window_step<16>(dkey2, v); }

  // persistent B operands: this lane's query row of Q1, Q2 (pre-multiplied by sm_scale*log2(e)
  // exactly as in the forward kernel, so the recomputed probabilities match it), dX, and its row
  // statistics
  h8 qf1[NKS], qf2[NKS], xf[NKV];
  {
    const float c = p.sm_scale * kLog2e;
    // a padding row stands in with the last real row, as in the forward; its results are not stored
    int qr = qt * BM + wave * 32 + j;
    if (TAIL && qr >= p.n_keys) qr = p.n_keys - 1;
    const half_t* r1 = p.q1 + qk_base + (size_t)qr * qk_n + 8 * g;
    const half_t* r2 = p.q2 + qk_base + (size_t)qr * qk_n + 8 * g;
    const half_t* rx = p.dx + qrow * DV + 8 * g;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      h8 a = *reinterpret_cast<const h8*>(r1 + 16 * ks);
      h8 b = *reinterpret_cast<const h8*>(r2 + 16 * ks);
#pragma unroll
      for (int e = 0; e < 8; ++e) { a[e] = (half_t)((float)a[e] * c); b[e] = (half_t)((float)b[e] * c); }
      qf1[ks] = a; qf2[ks] = b;
    }
#pragma unroll
    for (int kv = 0; kv < NKV; ++kv) xf[kv] = *reinterpret_cast<const h8*>(rx + 16 * kv);
  }
  const float nl1_ld = p.stat[0 * rows + qrow], nl2_ld = p.stat[1 * rows + qrow];
  const float de1_ld = p.stat[2 * rows + qrow], de2_ld = p.stat[3 * rows + qrow];

  f16v dq1[NDT], dq2[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) { dq1[t][r] = 0.f; dq2[t][r] = 0.f; }

  using KTile = AsyncTile<BN, D, NW>;
  using VTile = AsyncTile<BN, DV, NW>;
  const half_t* gk1 = p.k1 + qk_base;
  const half_t* gk2 = p.k2 + qk_base;
  const half_t* gv = p.v + v_base;
  const unsigned k_off = KTile::lane_off(wave, lane, qk_n), v_off = VTile::lane_off(wave, lane, v_n);
  // causal: keys beyond the last row of the workgroup are never visited
  // padding: tiles that hold no real key are not visited either
  // (an even count in every variant: with padding, a last tile without a real key may be visited; its keys are masked)
  const int n_tiles = CAUSAL ? (qt + 1) * (BM / BN) : PADDED ? (((p.n_keys + BN - 1) / BN + 1) & ~1) : p.N / BN;
  constexpr int VH = (VTile::PER + 1) / 2;

  // loads a wave issues per iteration (one K1, one K2 and one V tile)
  const int loads_per_iter = 2 * KTile::count(wave) + VTile::count(wave);
  // with padding, the tiles that reach past the last real key are copied with their row index clamped to it
  auto copy_k = [&](const half_t* gk, int t, lds_half* dst) {
    if (TAIL && (t + 1) * BN > p.n_keys) KTile::issue_clamped(gk + (size_t)t * BN * qk_n, dst, wave, lane, k_off, qk_n, p.n_keys - 1 - t * BN);
    else KTile::issue_at(gk + (size_t)t * BN * qk_n, dst, wave, lane, k_off, qk_n);
  };
  auto copy_v = [&](int t, lds_half* dst, auto k0_tag, auto k1_tag) {
    constexpr int K0 = decltype(k0_tag)::value, K1 = decltype(k1_tag)::value;
    if (TAIL && (t + 1) * BN > p.n_keys) VTile::template issue_clamped<K0, K1>(gv + (size_t)t * BN * v_n, dst, wave, lane, v_off, v_n, p.n_keys - 1 - t * BN);
    else VTile::template issue_at<K0, K1>(gv + (size_t)t * BN * v_n, dst, wave, lane, v_off, v_n);
  };
  constexpr std::integral_constant<int, 0> v_begin{};
  constexpr std::integral_constant<int, VH> v_mid{};
  constexpr std::integral_constant<int, VTile::PER> v_end{};
  // tile memory by kind: K1 and K2 of buffer b, then the V tiles
  auto k_buf = [&](int b) { return smem + b * (C::KBUF_BYTES / 2); };
  auto v_buf = [&](int b) { return smem + C::VBASE_BYTES / 2 + b * C::V_TILE; };
  auto fetch_all = [&](int t, int buf) {
    copy_k(gk1, t, k_buf(buf));
    copy_k(gk2, t, k_buf(buf) + C::K_TILE);
    copy_v(t, v_buf(buf), v_begin, v_end);
  };
  // The loop runs whole turns of the ring (NBUF iterations); the tile count is even, so when it is not a
  // multiple of four, half a turn comes first and tile 0 goes into buffer 2: tile t is in buffer (t + b0) % NBUF.
  static_assert(C::NBUF == 4, "the loop is unrolled over a ring of four");
  const bool head_half = (n_tiles & 2) != 0;
  const int b0 = head_half ? 2 : 0;
  fetch_all(0, b0);
  fetch_all((n_tiles > 1) ? 1 : 0, b0 + 1);
  if constexpr (kPipe) fetch_all((n_tiles > 2) ? 2 : n_tiles - 1, (b0 + 2) % C::NBUF);   // it fetches three tiles ahead
  // dX and the row statistics are first used inside the loop, and the compiler waits for a load where it is first
  // used.  It does not see the asynchronous tile copies, so its wait for "the newest loads" would in fact be a
  // wait for every tile copy in flight, in every iteration.  Touching the registers here puts that wait in front
  // of the loop, where the first tiles are waited for anyway.
  // The pipelined form runs one wave per SIMD, and for a kernel with that register budget the compiler selects
  // every MFMA with its C and D operands in AGPRs: right for the dQ accumulators, but each recomputed score
  // and dP value then costs a copy back for the element-wise work (a quarter of the loop's VALU instructions).
  // There the three score products are issued as assembly with their results in VGPRs and the resident
  // Q1, Q2 and dX rows, which are only ever B operands, in AGPRs.  (Not in the dropout instantiations, whose
  // mask arithmetic makes the compiler move operands about: see bwd_dkdv_kernel.)
  if constexpr (kPipe) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) { keep_in_agpr(qf1[ks]); keep_in_agpr(qf2[ks]); }
#pragma unroll
    for (int kv = 0; kv < NKV; ++kv) keep_in_agpr(xf[kv]);
  } else {
#pragma unroll
    for (int kv = 0; kv < NKV; ++kv) asm volatile("" : "+v"(xf[kv]));
  }
  float nl1 = nl1_ld, nl2 = nl2_ld, de1 = de1_ld, de2 = de2_ld;
  asm volatile("" : "+v"(nl1), "+v"(nl2), "+v"(de1), "+v"(de2));
  if (C::PAIR || kPipe) wait_async_tiles();         // tiles 0 and 1 are read before the next barrier
  else wait_async_tiles_except(loads_per_iter);     // tile 0 has landed, tile 1 may still be in flight
  __syncthreads();

  // Per-lane LDS byte addresses, computed once.  The XOR swizzle makes the address of a fragment a different
  // function of the lane for every 16-byte chunk column, so there is one register per chunk column a lane
  // reads; the ring buffer, K1 or K2, the 32-key sub-tile and the k-step of 16 keys are multiples of 16 rows,
  // which the swizzle does not see, and travel in the instructions' immediate offsets.
  const int tr_row = 4 * g + ((lane & 15) >> 2);
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const unsigned lds0 = (unsigned)(unsigned long)smem;
  unsigned kfr[NKS], vfr[NKV], ktr[NDT][2];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) kfr[ks] = lds0 + 2u * (unsigned)swz_off<D>(j, 16 * ks + 8 * g);
#pragma unroll
  for (int kv = 0; kv < NKV; ++kv) vfr[kv] = lds0 + C::VBASE_BYTES + 2u * (unsigned)swz_off<DV>(j, 16 * kv + 8 * g);
#pragma unroll
  for (int tt = 0; tt < NDT; ++tt)
#pragma unroll
    for (int e = 0; e < 2; ++e) ktr[tt][e] = lds0 + 2u * (unsigned)swz_off<D>(tr_row + 8 * e, 32 * tt + tr_col);
  // kept as they are: the compiler neither folds constants into them nor recomputes them in the loop
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(kfr[ks]));
#pragma unroll
  for (int kv = 0; kv < NKV; ++kv) asm volatile("" : "+v"(vfr[kv]));
#pragma unroll
  for (int tt = 0; tt < NDT; ++tt) asm volatile("" : "+v"(ktr[tt][0]), "+v"(ktr[tt][1]));

  // Where registers allow, a row statistic that is added to every element of a product is the product's
  // initial accumulator value instead: sixteen registers that hold it, for sixteen additions less per sub-tile.
  constexpr bool kFoldDP = !DROP && (D == 32 || (D == 64 && (MASK == 0 || PIPE)));     // dP starts from -delta1 (not with dropout, which masks dP first)
  constexpr bool kFoldS = (D == 32);       // S1, S2 start from the negated logsumexp
  f16v de1v, nl1v, nl2v;
#pragma unroll
  for (int r = 0; r < 16; ++r) { de1v[r] = kFoldDP ? de1 : 0.f; nl1v[r] = kFoldS ? nl1 : 0.f; nl2v[r] = kFoldS ? nl2 : 0.f; }
  if constexpr (kFoldDP) asm volatile("" : "+v"(de1v));
  if constexpr (kFoldS) asm volatile("" : "+v"(nl1v), "+v"(nl2v));

  if constexpr (kPipe) {
    // One wave per SIMD has nobody to run its element-wise work under, so the loop is pipelined inside the wave,
    // as in the dK/dV kernel: while the element-wise work of 32-key sub-tile i runs on the VALU, row by row, the
    // score products of sub-tile i+1 (assembly, results in VGPRs) run on the matrix unit; the dQ products of
    // sub-tile i follow.  The workgroup meets once per tile, in the step that scores the tile's first sub-tile; that
    // step requests the tile after the next.
    struct Scores { f16v s1, s2, dp; };
    constexpr int SPT = BN / 32, RING = SPT * C::NBUF, HALF = RING / 2;   // sub-tiles per tile, steps per turn of the ring
    constexpr int NPROD = 2 * NKS + NKV;              // score products per sub-tile: S1 and S2 alternating, then dP
    // A fragment of product k of the sub-tile at byte offsets (KOFF, VOFF)
    auto prod_frag = [&](auto koff_tag, auto voff_tag, int k) -> h8 {
      constexpr int KOFF = decltype(koff_tag)::value, VOFF = decltype(voff_tag)::value;
      if (k < 2 * NKS) return lds_read_at<h8>(kfr[k / 2], KOFF + (k & 1) * C::K_TILE * 2);
      return lds_read_at<h8>(vfr[k - 2 * NKS], VOFF);
    };
    auto prod_mfma = [&](int k, h8 a, Scores& s) {
      if (k < 2) {
        if (k) s.s2 = kFoldS ? mfma32_bagpr_from(a, qf2[0], nl2v) : mfma32_bagpr_first(a, qf2[0]);
        else   s.s1 = kFoldS ? mfma32_bagpr_from(a, qf1[0], nl1v) : mfma32_bagpr_first(a, qf1[0]);
      } else if (k < 2 * NKS) {
        const int ks = k / 2;
        if (k & 1) s.s2 = mfma32_bagpr(a, qf2[ks], s.s2);
        else       s.s1 = mfma32_bagpr(a, qf1[ks], s.s1);
      } else if (k == 2 * NKS) {
        s.dp = kFoldDP ? mfma32_bagpr_from(a, xf[0], de1v) : mfma32_bagpr_first(a, xf[0]);
      } else {
        s.dp = mfma32_bagpr(a, xf[k - 2 * NKS], s.dp);
      }
    };
    constexpr int DEPTH = 4;                          // A fragments requested ahead of their product
    Scores sa, sb;
    {
      // scores of sub-tile 0, nothing to run them under
      h8 a[NPROD];
      if (head_half) {
#pragma unroll
        for (int k = 0; k < NPROD; ++k)
          a[k] = prod_frag(std::integral_constant<int, 2 * C::KBUF_BYTES>{}, std::integral_constant<int, 2 * C::VBUF_BYTES>{}, k);
      } else {
#pragma unroll
        for (int k = 0; k < NPROD; ++k) a[k] = prod_frag(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, k);
      }
#pragma unroll
      for (int k = 0; k < NPROD; ++k) prod_mfma(k, a[k], sa);
      mfma_results_ready(sa.s1, sa.s2, sa.dp);
    }

    auto step = [&](int i, auto pos_tag, Scores& cur, Scores& nxt) {
      constexpr int POS = decltype(pos_tag)::value, PNXT = (POS + 1) % RING;
      constexpr int BNXT = PNXT / SPT, BFAR = (BNXT + 2) % C::NBUF;
      constexpr bool opens = (PNXT % SPT) == 0;       // this step scores the first sub-tile of a tile
      constexpr int KCUR = (POS / SPT) * C::KBUF_BYTES + (POS % SPT) * 32 * D * 2;
      constexpr std::integral_constant<int, BNXT * C::KBUF_BYTES + (PNXT % SPT) * 32 * D * 2> knext{};
      constexpr std::integral_constant<int, BNXT * C::VBUF_BYTES + (PNXT % SPT) * 32 * DV * 2> vnext{};
      const int t3 = i / SPT + 3, tf = t3 < n_tiles ? t3 : n_tiles - 1;   // past the end: harmless re-reads
      if constexpr (opens) {
        // that tile has landed for everybody, and every wave is done with the tile whose buffer is refilled now
        wait_async_tiles_except(loads_per_iter);
        __syncthreads();
        copy_k(gk1, tf, k_buf(BFAR));
      }
      if constexpr (CAUSAL) {
        // only the last sub-tiles of a wave's loop reach past its first row: mask key > query there
        const int wrow0 = qt * BM + wave * 32;
        const int kbase = i * 32;
        if (kbase + 31 > wrow0) {
          const int rel = wrow0 + j - kbase - 4 * g;     // query index minus the key index of register 0
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (8 * (r / 4) + (r % 4) > rel) { cur.s1[r] = -INFINITY; cur.s2[r] = -INFINITY; }
        }
      }
      if constexpr (PADDED) {
        const int kbase = i * 32;
        if (kbase + 32 > p.n_keys) {
          const int rel = p.n_keys - 1 - kbase - 4 * g;   // last real key minus the key index of register 0
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (8 * (r / 4) + (r % 4) > rel) { cur.s1[r] = -INFINITY; cur.s2[r] = -INFINITY; }
        }
      }
      // the transposed K fragments of this sub-tile's dQ products are requested here and arrive under the loop below
      h8 tk1[2][NDT], tk2[2][NDT];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int tt = 0; tt < NDT; ++tt) {
          const int off = KCUR + 16 * kk * D * 2;
          tk1[kk][tt] = join(lds_read_tr_at(ktr[tt][0], off), lds_read_tr_at(ktr[tt][1], off));
          tk2[kk][tt] = join(lds_read_tr_at(ktr[tt][0], off + C::K_TILE * 2), lds_read_tr_at(ktr[tt][1], off + C::K_TILE * 2));
        }
      h8 a[NPROD];
#pragma unroll
      for (int k = 0; k < DEPTH; ++k) a[k] = prod_frag(knext, vnext, k);
      h8 b1[2], b2[2];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < NPROD; ++k) {
        if (k + DEPTH < NPROD) a[k + DEPTH] = prod_frag(knext, vnext, k + DEPTH);
        // the far tile's copies are spread over the products
        if (opens && k == NPROD / 4) copy_k(gk2, tf, k_buf(BFAR) + C::K_TILE);
        if (opens && k == NPROD / 2) copy_v(tf, v_buf(BFAR), v_begin, v_mid);
        if (opens && k == 3 * NPROD / 4) copy_v(tf, v_buf(BFAR), v_mid, v_end);
        prod_mfma(k, a[k], nxt);
        // element-wise rows of this sub-tile, spread evenly over the products
        const int r0 = 16 * k / NPROD, r1 = 16 * (k + 1) / NPROD;
#pragma unroll
        for (int r = r0; r < r1; ++r) {
          const float p1 = fast_exp2(kFoldS ? cur.s1[r] : cur.s1[r] + nl1);
          const float p2 = fast_exp2(kFoldS ? cur.s2[r] : cur.s2[r] + nl2);
          // in fp32 up to the rounding of dS itself (see the loop of the other head dims)
          const float dpc = kFoldDP ? cur.dp[r] : cur.dp[r] + de1;
          b1[r / 8][r % 8] = (half_t)(p1 * dpc);
          b2[r / 8][r % 8] = (half_t)(p2 * __builtin_fmaf(-lam, dpc, de2));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      mfma_results_ready(nxt.s1, nxt.s2, nxt.dp);     // the next step's VALU reads them
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int tt = 0; tt < NDT; ++tt) {
          dq1[tt] = mfma32(tk1[kk][tt], b1[kk], dq1[tt]);
          dq2[tt] = mfma32(tk2[kk][tt], b2[kk], dq2[tt]);
        }
    };

    auto half_turn = [&](int i, auto h0_tag) {
      constexpr int H0 = decltype(h0_tag)::value;
      step(i, std::integral_constant<int, H0>{}, sa, sb);
      step(i + 1, std::integral_constant<int, H0 + 1>{}, sb, sa);
      if constexpr (HALF == 4) {
        step(i + 2, std::integral_constant<int, H0 + 2>{}, sa, sb);
        step(i + 3, std::integral_constant<int, H0 + 3>{}, sb, sa);
      }
    };
    const int n_steps = n_tiles * SPT;
    int i = 0;
    if (head_half) {
      half_turn(0, std::integral_constant<int, HALF>{});
      i = HALF;
    }
#pragma nounroll
    for (; i < n_steps; i += RING) {
      half_turn(i, std::integral_constant<int, 0>{});
      half_turn(i + HALF, std::integral_constant<int, HALF>{});
    }
  } else {
  // One iteration: tile t, in the buffer at ring position POS; tile t+2 is requested into the buffer two
  // positions on, which held a tile that every wave has finished reading.
  auto iteration = [&](int t, auto pos_tag) {
    constexpr int POS = decltype(pos_tag)::value;
    constexpr int KCUR = POS * C::KBUF_BYTES, VCUR = POS * C::VBUF_BYTES, BNXT = (POS + 2) % C::NBUF;
    const int tn = (t + 2 < n_tiles) ? t + 2 : n_tiles - 1;   // past the end: harmless re-reads
    copy_k(gk1, tn, k_buf(BNXT));

#pragma unroll
    for (int ksub = 0; ksub < BN / 32; ++ksub) {
      if (ksub == 0) copy_k(gk2, tn, k_buf(BNXT) + C::K_TILE);
      // transposed tiles [32 keys x 32 queries]: this lane's column is its query
      f16v s1 = nl1v, s2 = nl2v, dp = de1v;       // zero, or the folded statistic
      // all fragments of the three score products are requested before the first product is issued
      h8 ak1[NKS], ak2[NKS], av[NKV];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        ak1[ks] = lds_read_at<h8>(kfr[ks], KCUR + ksub * 32 * D * 2);
        ak2[ks] = lds_read_at<h8>(kfr[ks], KCUR + C::K_TILE * 2 + ksub * 32 * D * 2);
      }
#pragma unroll
      for (int kv = 0; kv < NKV; ++kv) av[kv] = lds_read_at<h8>(vfr[kv], VCUR + ksub * 32 * DV * 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        s1 = mfma32(ak1[ks], qf1[ks], s1);
        s2 = mfma32(ak2[ks], qf2[ks], s2);
      }
#pragma unroll
      for (int kv = 0; kv < NKV; ++kv) dp = mfma32(av[kv], xf[kv], dp);
      if (ksub == 0) copy_v(tn, v_buf(BNXT), v_begin, v_mid);
      // with a barrier every second tile all of a tile's copies go out early: they have to land by the next barrier
      if (ksub == (C::PAIR ? 0 : BN / 32 - 1)) copy_v(tn, v_buf(BNXT), v_mid, v_end);
      if constexpr (CAUSAL) {
        // only the last sub-tiles of a wave's loop reach past its first row: mask key > query there
        const int wrow0 = qt * BM + wave * 32;
        const int kbase = t * BN + ksub * 32;
        if (kbase + 31 > wrow0) {
          const int rel = wrow0 + j - kbase - 4 * g;     // query index minus the key index of register 0
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (8 * (r / 4) + (r % 4) > rel) { s1[r] = -INFINITY; s2[r] = -INFINITY; }
        }
      }
      if constexpr (PADDED) {
        // only the last sub-tiles hold padding keys
        const int kbase = t * BN + ksub * 32;
        if (kbase + 32 > p.n_keys) {
          const int rel = p.n_keys - 1 - kbase - 4 * g;   // last real key minus the key index of register 0
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (8 * (r / 4) + (r % 4) > rel) { s1[r] = -INFINITY; s2[r] = -INFINITY; }
        }
      }
      // The transposed K fragments of the dQ products do not depend on the element-wise work: they
      // are requested before it and arrive while it runs.  (Left to itself the compiler requests
      // each one right in front of its product and waits out the LDS latency eight times.)
      // (The dropout instantiations need the registers for the mask arithmetic and read each
      // fragment in front of its product instead.)
      h8 tk1[2][NDT], tk2[2][NDT];
      auto read_tk = [&](int kk, int tt) {
        const int off = KCUR + (ksub * 32 + 16 * kk) * D * 2;
        tk1[kk][tt] = join(lds_read_tr_at(ktr[tt][0], off), lds_read_tr_at(ktr[tt][1], off));
        tk2[kk][tt] = join(lds_read_tr_at(ktr[tt][0], off + C::K_TILE * 2), lds_read_tr_at(ktr[tt][1], off + C::K_TILE * 2));
      };
      constexpr bool kFragmentsAhead = !DROP;
      if constexpr (kFragmentsAhead) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int tt = 0; tt < NDT; ++tt) read_tk(kk, tt);
      }
      __builtin_amdgcn_sched_barrier(0);
      h8 b1[2], b2[2];
      unsigned w1 = 0, w2 = 0, w1b = 0, w2b = 0;
      const unsigned hkeys = hrow + (unsigned)(t * (BN / 2) + ksub * 16);
      const unsigned hwin1 = DROP ? dropout_window<16>(dkey1, hkeys, hlow) : 0u;
      const unsigned hwin2 = DROP ? dropout_window<16>(dkey2, hkeys, hlow) : 0u;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p1 = fast_exp2(kFoldS ? s1[r] : s1[r] + nl1);
        const float p2 = fast_exp2(kFoldS ? s2[r] : s2[r] + nl2);
        if constexpr (DROP) {
          // register r holds key 8*(r/4) + 4g + (r%4) of the sub-tile; registers r, r+1 (r even) share the hash words
          // of their 2x2 block, and the blocks of registers r..r+1 and r+2..r+3 (r a multiple of 4) are neighbours,
          // hashed one by each lane of a query pair
          if ((r & 3) == 0) {
            dropout_bytes_shared(dropout_rounds(dkey1, hwin1 + hstep1[r / 4]), dsel, w1, w1b);
            dropout_bytes_shared(dropout_rounds(dkey2, hwin2 + hstep2[r / 4]), dsel, w2, w2b);
          }
          // the probabilities carry c, statistics 2 and 3 are -delta1/c and -delta2/c
          const float d1 = dropout_keep_half((r & 2) ? w1b : w1, r & 1, p.drop.threshold) ? dp[r] : 0.f;
          const float d2 = dropout_keep_half((r & 2) ? w2b : w2, r & 1, p.drop.threshold) ? dp[r] : 0.f;
          b1[r / 8][r % 8] = (half_t)(p1 * (d1 + de1));                         // c A1 (m1 dP - delta1/c)
          b2[r / 8][r % 8] = (half_t)(p2 * __builtin_fmaf(-lam, d2, de2));      // c A2 (-lambda m2 dP - delta2/c)
        } else {
          // in fp32 up to the rounding of dS itself: dP - delta alone may exceed the 16-bit range when the
          // upstream gradient carries a loss scale, while its product with the probability does not
          const float dpc = kFoldDP ? dp[r] : dp[r] + de1;                  // statistic 2 is -delta1
          b1[r / 8][r % 8] = (half_t)(p1 * dpc);
          b2[r / 8][r % 8] = (half_t)(p2 * __builtin_fmaf(-lam, dpc, de2));   // statistic 3 is -(lambda*delta1 + delta2)
        }
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int tt = 0; tt < NDT; ++tt) {
          if constexpr (!kFragmentsAhead) read_tk(kk, tt);
          dq1[tt] = mfma32(tk1[kk][tt], b1[kk], dq1[tt]);
          dq2[tt] = mfma32(tk2[kk][tt], b2[kk], dq2[tt]);
        }
    }

    if constexpr (C::PAIR) {
      // Every second tile the workgroup meets: the copies of the next two tiles (requested during the last
      // two) have landed for everybody, and the buffers of the last two tiles may be refilled.
      if constexpr (POS & 1) {
        wait_async_tiles();
        __syncthreads();
      }
    } else {
      // tile t+1 was requested one iteration ago: only this iteration's loads may remain in flight
      wait_async_tiles_except(loads_per_iter);
      __syncthreads();
    }
  };

  int t = 0;
  if (head_half) {
    iteration(0, std::integral_constant<int, 2>{});
    iteration(1, std::integral_constant<int, 3>{});
    t = 2;
  }
#pragma nounroll
  for (; t < n_tiles; t += 4) {
    iteration(t, std::integral_constant<int, 0>{});
    iteration(t + 1, std::integral_constant<int, 1>{});
    iteration(t + 2, std::integral_constant<int, 2>{});
    iteration(t + 3, std::integral_constant<int, 3>{});
  }
  }
  wait_async_tiles();
  __syncthreads();      // the tile memory is reused below; other waves may still have been reading it

  // dQ^T tile tt: this lane's column is its query; register r = feature 32*tt + 8*(r/4) + 4g + (r%4).
  // The accumulated sums carry log2(e) from the pre-scaled Q only inside the probabilities, so the
  // remaining factor is the plain softmax scale.  Each wave stages its 32 rows of dQ1 and dQ2 in the
  // now idle tile memory (8 bytes per lane, row stride D+8 halfs) and reads them back row by row, so
  // that the global stores are whole 16-byte chunks of consecutive rows.
  constexpr int SROW = D + 8;
  static_assert(NW * 2 * 32 * SROW <= C::NBUF * C::STAGE, "staging blocks fit the tile memory");
  lds_half* const stg = smem + (size_t)wave * 2 * 32 * SROW;
#pragma unroll
  for (int tt = 0; tt < NDT; ++tt)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      h4 v1, v2;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v1[e] = (half_t)(dq1[tt][4 * r4 + e] * p.sm_scale);
        v2[e] = (half_t)(dq2[tt][4 * r4 + e] * p.sm_scale);
      }
      *(DA_LDS h4*)(stg + j * SROW + 32 * tt + 8 * r4 + 4 * g) = v1;
      *(DA_LDS h4*)(stg + (32 + j) * SROW + 32 * tt + 8 * r4 + 4 * g) = v2;
    }
  __builtin_amdgcn_wave_barrier();   // the rows are read back by other lanes of this wave only
  constexpr int LPR = D / 8;         // lanes per row
  constexpr int RPI = 64 / LPR;      // rows per instruction
  const int qloc0 = qt * BM + wave * 32;             // first query of this wave inside the unit
  const size_t ob = da_abi::unit_base(p, p.sdqk, bh) + (size_t)qloc0 * (size_t)p.sdqk.n;
  half_t* const o1 = p.dq1 + ob;
  half_t* const o2 = p.dq2 + ob;
#pragma unroll
  for (int k = 0; k < 32 / RPI; ++k) {
    const int row = k * RPI + lane / LPR, ch = lane % LPR;
    const u32x4 v1 = *(const DA_LDS u32x4*)(stg + row * SROW + 8 * ch);
    const u32x4 v2 = *(const DA_LDS u32x4*)(stg + (32 + row) * SROW + 8 * ch);
    if (!TAIL || qloc0 + row < p.n_keys) {    // the gradient tensors have no rows past the real length
      *reinterpret_cast<u32x4*>(o1 + (size_t)row * (size_t)p.sdqk.n + 8 * ch) = v1;
      *reinterpret_cast<u32x4*>(o2 + (size_t)row * (size_t)p.sdqk.n + 8 * ch) = v2;
    }
  }
}

template <int D, int NWAVES, int MASK, bool DROP>
__global__ __launch_bounds__((DqCfg<D, NWAVES, false>::REG_NT)) __attribute__((amdgpu_waves_per_eu(DqCfg<D, NWAVES, false>::OCC, DqCfg<D, NWAVES, false>::OCC)))
void bwd_dq_kernel(BwdParams p) {
  using C = DqCfg<D, NWAVES, false>;
  __shared__ __attribute__((aligned(16))) half_t smem[C::SMEM];
  static_assert(sizeof(smem) >= 256 * sizeof(float), "the hosted reduction uses the tile memory");
  DA_HOST_DLAMBDA(smem)
  dq_block<D, NWAVES, MASK, DROP, false>(p, blockIdx.x, gridDim.x - p.dlam_fold, (lds_half*)smem);
}

// dK/dV blocks and dQ blocks in one grid: the two have nothing to wait for in each other, and as launches of their
// own each leaves the CUs that its last (or only) round of workgroups does not reach idle.  All blocks are four
// waves at one wave per SIMD, the long ones first: p.n_kv_wg key blocks (at D = 128 twice, for dK and for dV), then
// p.n_q_wg query blocks.  Measured against separate launches (whole backward, N(0,1) fp16): B1 H16 N128 D128 49 -> 25 us,
// B2 H16 N512 D64 48 -> 33, B1 H8 N2048 D64 121 -> 80 (causal 134 -> 73), B1 H12 N3584 D128 848 -> 648,
// B8 H32 N4096 D128 18.5 -> 18.3 ms.
template <int D, bool CAUSAL, bool PADDED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_pair_kernel(BwdParams p) {
  constexpr int SK = DkvCfg<D, CAUSAL>::SMEM, SQ = DqCfg<D, 4, true>::SMEM;
  static_assert(DkvCfg<D, false>::NT == 256, "both kinds of blocks have four waves");
  __shared__ __attribute__((aligned(16))) half_t smem[SK > SQ ? SK : SQ];
  DA_HOST_DLAMBDA(smem)
  int wg = blockIdx.x;
  const int n_kv = p.n_kv_wg;
  if (wg < n_kv) {
    dkdv_block<D, D == 128 ? 2 : 0, CAUSAL, false, PADDED>(p, wg, n_kv, (lds_half*)smem);
    return;
  }
  wg -= n_kv;
  if constexpr (D == 128) {
    if (wg < n_kv) {
      dkdv_block<D, 1, CAUSAL, false, PADDED>(p, wg, n_kv, (lds_half*)smem);
      return;
    }
    wg -= n_kv;
  }
  dq_block<D, 4, CAUSAL ? 1 : PADDED ? 2 : 0, false, true>(p, wg, p.n_q_wg, (lds_half*)smem);
}

template <int D>
static hipError_t launch_bwd_t(const BwdParams& p_in, hipStream_t stream) {
  BwdParams p = p_in;
  const int n_prep = bwd_num_partials(p.BH, p.N, D);
  hipError_t e = hipSuccess;
  // the d(lambda) reduce rides in the first dK/dV or dQ launch when there is one, else it is a launch of its own
  const int n_lambda = p.lambda_stride ? p.H : 1;
  bool fold = (p.stages & 2u) && (p.stages & 12u);
  p.dlam_fold = 0;
  if (p.stages & 1u) {
    if (p.gain)         // of normalised heads
      hipLaunchKernelGGL((bwd_prep_kernel<D, true, true>), dim3(n_prep), dim3(256), 0, stream, p);
    else if (p.rms_norm)
      hipLaunchKernelGGL((bwd_prep_kernel<D, true>), dim3(n_prep), dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((bwd_prep_kernel<D, false>), dim3(n_prep), dim3(256), 0, stream, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if ((p.stages & 2u) && !fold) {
    hipLaunchKernelGGL(bwd_dlambda_kernel, dim3(n_lambda), dim3(256), 0, stream,
                       p.dlam_part, n_prep / p.BH, p.BH, p.dlambda, p.lambda_fp32);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (!(p.stages & 12u)) return e;
  const bool padded = p.n_keys < p.N;
  if (da_abi::bwd_one_grid(D, p.drop.threshold != 0, p.causal, p.N, (long long)p.BH * (p.N / 128), p.stages)) {
    const int blocks = p.BH * (p.N / 128);
    p.n_kv_wg = (p.stages & 4u) ? blocks : 0;
    p.n_q_wg = (p.stages & 8u) ? blocks : 0;
    p.dlam_fold = fold ? n_lambda : 0;
    const dim3 grid((D == 128 ? 2 : 1) * p.n_kv_wg + p.n_q_wg + p.dlam_fold), block(256);
    if (p.causal) {
      if (padded) hipLaunchKernelGGL((bwd_pair_kernel<D, true, true>), grid, block, 0, stream, p);
      else        hipLaunchKernelGGL((bwd_pair_kernel<D, true, false>), grid, block, 0, stream, p);
    } else {
      if (padded) hipLaunchKernelGGL((bwd_pair_kernel<D, false, true>), grid, block, 0, stream, p);
      else        hipLaunchKernelGGL((bwd_pair_kernel<D, false, false>), grid, block, 0, stream, p);
    }
    return hipGetLastError();
  }
  if (p.stages & 4u) {
    const dim3 block(DkvCfg<D, false>::NT);
    auto launch_mode = [&](auto mode_tag) {
      constexpr int M = decltype(mode_tag)::value;
      p.dlam_fold = fold ? n_lambda : 0;
      fold = false;
      const dim3 grid(p.BH * (p.N / DkvCfg<D, false>::BK) + p.dlam_fold);
      auto launch_padded = [&](auto padded_tag) {
        constexpr bool PAD = decltype(padded_tag)::value;
        if (p.drop.threshold) {
          if (p.causal) hipLaunchKernelGGL((bwd_dkdv_kernel<D, M, true, true, PAD>), grid, block, 0, stream, p);
          else          hipLaunchKernelGGL((bwd_dkdv_kernel<D, M, false, true, PAD>), grid, block, 0, stream, p);
        } else if constexpr (D != 128) {
          if (p.causal) hipLaunchKernelGGL((bwd_dkdv_kernel<D, M, true, false, PAD>), grid, block, 0, stream, p);
          else          hipLaunchKernelGGL((bwd_dkdv_kernel<D, M, false, false, PAD>), grid, block, 0, stream, p);
        }
      };
      if (padded) launch_padded(std::true_type{});
      else        launch_padded(std::false_type{});
    };
    if constexpr (D == 128) {
      launch_mode(std::integral_constant<int, 1>{});
      if ((e = hipGetLastError()) != hipSuccess) return e;
      launch_mode(std::integral_constant<int, 2>{});
    } else {
      launch_mode(std::integral_constant<int, 0>{});
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (p.stages & 8u) {
    // 256 query rows per workgroup when the sequence allows it, otherwise 128 (a D = 128 workgroup
    // runs one wave per SIMD and therefore always has four waves).  A grid so small that even its
    // 128-row workgroups all fit on the chip at once is launched that way too: it finishes sooner
    // in twice as many, half as long workgroups.
    auto launch_dq = [&](auto nw_tag) {
      constexpr int NWV = decltype(nw_tag)::value;
      p.dlam_fold = fold ? n_lambda : 0;
      fold = false;
      const dim3 grid(p.BH * (p.N / (32 * NWV)) + p.dlam_fold), block(64 * NWV);
      if (p.drop.threshold) {
        if (p.causal)    hipLaunchKernelGGL((bwd_dq_kernel<D, NWV, 1, true>), grid, block, 0, stream, p);
        else if (padded) hipLaunchKernelGGL((bwd_dq_kernel<D, NWV, 2, true>), grid, block, 0, stream, p);
        else             hipLaunchKernelGGL((bwd_dq_kernel<D, NWV, 0, true>), grid, block, 0, stream, p);
      } else if constexpr (D == 32 || (D == 64 && NWV == 8)) {      // the others go into one grid
        if (p.causal)    hipLaunchKernelGGL((bwd_dq_kernel<D, NWV, 1, false>), grid, block, 0, stream, p);
        else if (padded) hipLaunchKernelGGL((bwd_dq_kernel<D, NWV, 2, false>), grid, block, 0, stream, p);
        else             hipLaunchKernelGGL((bwd_dq_kernel<D, NWV, 0, false>), grid, block, 0, stream, p);
      }
    };
    if constexpr (D == 128) {
      launch_dq(std::integral_constant<int, 4>{});
    } else {
      // without dropout only grids of more than 256 128-row blocks come here
      if (p.N % 256 == 0 && (!p.drop.threshold || (long long)p.BH * (p.N / 128) > 256)) launch_dq(std::integral_constant<int, 8>{});
      else launch_dq(std::integral_constant<int, 4>{});
    }
  }
  return hipGetLastError();
}

hipError_t launch_bwd(const BwdParams& p, int D, hipStream_t stream) {
  switch (D) {
    case 32:  return launch_bwd_t<32>(p, stream);
    case 64:  return launch_bwd_t<64>(p, stream);
    case 128: return launch_bwd_t<128>(p, stream);
    default:  return hipErrorInvalidValue;
  }
}

}  // namespace DA_NS
