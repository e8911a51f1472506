// Kernels of the layer around the operator (modules.DiffAttn; the reference stops at the operator, src/layers.py:10-26):
//
//   wgrad_kernel         the weight gradients of the four projections, dW = dY^T X summed over the tokens
//   wgrad_reduce_kernel  sum of the partial products where the tokens are split between workgroups
//   layer_pack_kernel    the three input projections' weights in one matrix, and lambda from its four vectors
//   layer_finish_kernel  the gradients of the head gain and of the four lambda vectors
#include <type_traits>

#include "layer.hpp"

namespace DA_NS {

using da_abi::LayerFinishParams;
using da_abi::LayerPackParams;
using da_abi::WgradParams;

// ---- weight gradients ---------------------------------------------------------------------------
// dW[o][i] = sum over tokens t of dY[t][o] X[t][i].  Both operands are stored with the contraction index, the token, as
// the slow one, so both fragments of a product come from row-major tiles through the transposing LDS read, in the same
// token order.  A workgroup of eight waves owns a 128 x 128 tile of one weight: 64-token slabs of both operands go to a ring
// of four LDS buffers, three slabs ahead; waves 0-3 take the first 32 tokens of a slab and waves 4-7 the last 32, each wave
// a 64 x 64 quarter (four fragments for four products), and the two halves meet in LDS at the end.  Two waves per SIMD
// hide each other's LDS reads without a second workgroup, whose tile would have to be added through memory.  Bound by the
// matrix unit where the grid fills the chip (E 2048, 16384 tokens, one weight: 145 us, 948 TFLOP/s; a library product of that
// size 165 us), by the start and end of its workgroups and the sum of the splits where it does not (E 512, one weight, with
// wgrad_reduce_kernel: 23 us at 8192 and at 16384 tokens, library 52 and 98; between E 1024 and 2048 also by a last round that is
// partly empty: four weights of E 1152, 324 tiles for 256 CUs, 8192 tokens 147 us = 591 TFLOP/s).
struct WgradCfg {
  static constexpr int TILE = da_abi::kWgradTile, BK = da_abi::kWgradSlab, NW = 8, NT = NW * 64, NBUF = 4;
  static constexpr int BUF = BK * TILE;                              // halfs of one operand's slab
  static constexpr int BBASE = NBUF * BUF * 2;                       // byte offset of the second operand's ring
  static constexpr int SMEM = 2 * NBUF * BUF;                        // halfs
  static_assert(NBUF * BUF * 2 <= 65536, "immediate offsets reach every buffer");
  static_assert(SMEM * 2 >= 4 * 64 * 64 * 4, "the exchange of the two halves fits the tile memory");
};

__global__ __launch_bounds__(WgradCfg::NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void wgrad_kernel(WgradParams p) {
  using C = WgradCfg;
  __shared__ __attribute__((aligned(16))) half_t smem_[C::SMEM];
  lds_half* const smem = (lds_half*)smem_;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, g = lane >> 5;
  const int kh = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;     // half of a slab, quarter of the tile

  // consecutive workgroups of one XCD share the rows' operand, tile by tile
  const int nt = p.E / C::TILE;
  int id = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = id % nt; id /= nt;
  const int to = id % nt; id /= nt;
  const int split = id % p.split.splits, job = id / p.split.splits;
  const half_t* const ga = (const half_t*)p.job[job].a + (size_t)to * C::TILE;
  const half_t* const gb = (const half_t*)p.job[job].b + (size_t)ti * C::TILE;
  const int lda = p.job[job].lda, ldb = p.job[job].ldb;

  const int s0 = split * p.split.slabs;
  const int n_all = (p.T + C::BK - 1) / C::BK;
  const int n = min(p.split.slabs, n_all - s0);                  // at least one

  using Slab = AsyncTile<C::BK, C::TILE, C::NW>;
  static_assert(Slab::kOneOffset && Slab::NINST % C::NW == 0, "one offset and one count for every wave");
  const unsigned a_off = Slab::lane_off(wave, lane, lda), b_off = Slab::lane_off(wave, lane, ldb);
  auto fetch = [&](int s, int buf) {
    const int sl = s0 + (s < n ? s : n - 1);                         // past the end: harmless re-reads
    const size_t t = (size_t)sl * C::BK;
    lds_half* const la = smem + buf * C::BUF;
    lds_half* const lb = smem + C::BBASE / 2 + buf * C::BUF;
    if ((sl + 1) * C::BK > p.T) {
      const int last = p.T - 1 - sl * C::BK;
      Slab::issue_clamped(ga + t * lda, la, wave, lane, a_off, lda, last);
      Slab::issue_clamped(gb + t * ldb, lb, wave, lane, b_off, ldb, last);
    } else {
      Slab::issue_at(ga + t * lda, la, wave, lane, a_off, lda);
      Slab::issue_at(gb + t * ldb, lb, wave, lane, b_off, ldb);
    }
  };
  constexpr int LOADS = 2 * Slab::PER;
  static_assert(2 * LOADS <= 8, "two slabs in flight are counted");

  // per-lane addresses of the transposing reads; buffer and 16-token step travel in the immediate offset
  const int tr_row = 32 * kh + 4 * g + ((lane & 15) >> 2);
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const unsigned lds0 = (unsigned)(unsigned long)smem;
  unsigned fa[2][2], fb[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      fa[x][e] = lds0 + 2u * (unsigned)swz_off<C::TILE>(tr_row + 8 * e, 64 * wm + 32 * x + tr_col);
      fb[x][e] = lds0 + C::BBASE + 2u * (unsigned)swz_off<C::TILE>(tr_row + 8 * e, 64 * wn + 32 * x + tr_col);
      asm volatile("" : "+v"(fa[x][e]), "+v"(fb[x][e]));
    }

  f16v acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0.f;

  fetch(0, 0); fetch(1, 1); fetch(2, 2);
  auto slab = [&](int s, auto buf_tag) {
    constexpr int BUF = decltype(buf_tag)::value;
    wait_async_tiles_except(2 * LOADS);           // slab s has landed for this wave, s+1 and s+2 may be in flight
    __syncthreads();                              // ... and for everybody; everybody is done with slab s-1
    if ((s0 + s + 1) * C::BK > p.T) {
      // tokens past the last one hold copies of it: they count as zero
      const int real = p.T - (s0 + s) * C::BK;
      DA_LDS u32x4* const za = (DA_LDS u32x4*)(smem + BUF * C::BUF);
      DA_LDS u32x4* const zb = (DA_LDS u32x4*)(smem + C::BBASE / 2 + BUF * C::BUF);
      for (int k = real * (C::TILE / 8) + tid; k < C::BUF / 8; k += C::NT) { za[k] = u32x4{0u, 0u, 0u, 0u}; zb[k] = u32x4{0u, 0u, 0u, 0u}; }
      __syncthreads();
    }
    fetch(s + 3, (BUF + 3) % C::NBUF);
    h8 a[2][2], b[2][2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int off = BUF * C::BUF * 2 + 16 * kk * C::TILE * 2;
        a[kk][x] = join(lds_read_tr_at(fa[x][0], off), lds_read_tr_at(fa[x][1], off));
        b[kk][x] = join(lds_read_tr_at(fb[x][0], off), lds_read_tr_at(fb[x][1], off));
      }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = mfma32(a[kk][x], b[kk][y], acc[x][y]);
  };
  int s = 0;
#pragma nounroll
  for (; s + 4 <= n; s += 4) {
    slab(s, std::integral_constant<int, 0>{});
    slab(s + 1, std::integral_constant<int, 1>{});
    slab(s + 2, std::integral_constant<int, 2>{});
    slab(s + 3, std::integral_constant<int, 3>{});
  }
  if (s < n) slab(s, std::integral_constant<int, 0>{});
  if (s + 1 < n) slab(s + 1, std::integral_constant<int, 1>{});
  if (s + 2 < n) slab(s + 2, std::integral_constant<int, 2>{});
  wait_async_tiles();
  __syncthreads();

  // the second half's sums join the first's: lane to lane, both hold the same elements
  float* const xch = reinterpret_cast<float*>(smem_) + (size_t)(wave & 3) * 64 * 64;
  if (kh == 1) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          f4v v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[x][y][4 * r4 + e];
          *reinterpret_cast<f4v*>(xch + (((x * 2 + y) * 4 + r4) * 64 + lane) * 4) = v;
        }
  }
  __syncthreads();
  if (kh == 1) return;
  const size_t row0 = (size_t)to * C::TILE + 64 * wm, col0 = (size_t)ti * C::TILE + 64 * wn;
  half_t* const out = (half_t*)p.job[job].out;
  float* const part = p.part + ((size_t)split * p.n_jobs + job) * p.E * p.E;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f4v v = *reinterpret_cast<const f4v*>(xch + (((x * 2 + y) * 4 + r4) * 64 + lane) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // accumulator tile: column j, register r = row 8*(r/4) + 4g + (r%4)
          const size_t at = (row0 + 32 * x + 8 * r4 + 4 * g + e) * p.E + col0 + 32 * y + j;
          const float sum = acc[x][y][4 * r4 + e] + v[e];
          if (p.split.splits == 1) out[at] = (half_t)sum;
          else part[at] = sum;
        }
      }
}

// eight values a thread, the splits added in their order
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(WgradParams p) {
  const size_t size = (size_t)p.E * p.E, at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
  const int job = blockIdx.y;
  if (at >= size) return;
  const float* src = p.part + job * size + at;
  f4v lo = *reinterpret_cast<const f4v*>(src), hi = *reinterpret_cast<const f4v*>(src + 4);
#pragma unroll 4
  for (int s = 1; s < p.split.splits; ++s) {
    src += p.n_jobs * size;
    lo += *reinterpret_cast<const f4v*>(src);
    hi += *reinterpret_cast<const f4v*>(src + 4);
  }
  h8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) { v[e] = (half_t)lo[e]; v[4 + e] = (half_t)hi[e]; }
  *reinterpret_cast<h8*>((half_t*)p.job[job].out + at) = v;
}

hipError_t launch_wgrad(const WgradParams& p, hipStream_t stream) {
  const int nt = p.E / da_abi::kWgradTile;
  hipLaunchKernelGGL(wgrad_kernel, dim3(p.n_jobs * p.split.splits * nt * nt), dim3(WgradCfg::NT), 0, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.split.splits == 1) return e;
  const size_t size = (size_t)p.E * p.E;
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)((size / 8 + 255) / 256), p.n_jobs), dim3(256), 0, stream, p);
  return hipGetLastError();
}

// ---- weights and lambda ---------------------------------------------------------------------------
// exp(q1.k1) and exp(q2.k2) of one lambda, formed by one wave
struct LambdaTerms { float e1, e2; };
__device__ __forceinline__ LambdaTerms lambda_terms(const diffattn_lambda_vectors& v, int o, int lane) {
  float s1 = 0.f, s2 = 0.f;
  for (int i = lane; i < v.d; i += 64) {
    const int at = o * v.d + i;
    s1 += v.q1[at] * v.k1[at];
    s2 += v.q2[at] * v.k2[at];
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) { s1 += __shfl_xor(s1, m, 64); s2 += __shfl_xor(s2, m, 64); }
  return {expf(s1), expf(s2)};
}

#ifndef DA_BF16       // it copies bytes: one build serves both types
// the last workgroup forms lambda, the others copy the three weights one after another (16 bytes a thread and turn)
__global__ __launch_bounds__(256) void layer_pack_kernel(LayerPackParams p) {
  if (blockIdx.x == gridDim.x - 1) {
    if (!p.lambda) return;
    const int lane = threadIdx.x & 63;
    for (int o = threadIdx.x >> 6; o < p.vec.n; o += 4) {
      const LambdaTerms t = lambda_terms(p.vec, o, lane);
      if (lane == 0) p.lambda[o] = t.e1 - t.e2 + p.lambda_init;
    }
    return;
  }
  const size_t chunks = p.weight_bytes / 16, step = (size_t)(gridDim.x - 1) * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < 3 * chunks; i += step) {
    const int w = i >= 2 * chunks ? 2 : i >= chunks ? 1 : 0;
    reinterpret_cast<u32x4*>(p.packed)[i] = reinterpret_cast<const u32x4*>(p.w[w])[i - w * chunks];
  }
}

hipError_t launch_layer_pack(const LayerPackParams& p, hipStream_t stream) {
  const size_t want = (3 * (p.weight_bytes / 16) + 255) / 256;
  hipLaunchKernelGGL(layer_pack_kernel, dim3((unsigned)(want < 2048 ? want : 2048) + 1), dim3(256), 0, stream, p);
  return hipGetLastError();
}
#endif

// ---- the last sums of a backward -----------------------------------------------------------------
// d(gain): workgroup b sums columns 16b .. 16b+15 of the partials, 64 rows of them at a time, then a tree in a fixed order.
// The last workgroup writes the gradients of the lambda vectors.
__global__ __launch_bounds__(256) void layer_finish_kernel(LayerFinishParams p) {
  __shared__ f4v red[256];
  const int tid = threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {
    if (!p.dlambda) return;
    const int lane = tid & 63;
    for (int o = tid >> 6; o < p.vec.n; o += 4) {
      const LambdaTerms t = lambda_terms(p.vec, o, lane);
      const float a = p.dlambda[o] * t.e1, b = -p.dlambda[o] * t.e2;
      for (int i = lane; i < p.vec.d; i += 64) {
        const int at = o * p.vec.d + i;
        p.dq1[at] = a * p.vec.k1[at];
        p.dk1[at] = a * p.vec.q1[at];
        p.dq2[at] = b * p.vec.k2[at];
        p.dk2[at] = b * p.vec.q2[at];
      }
    }
    return;
  }
  const int col = 16 * blockIdx.x + 4 * (tid & 3), slot = tid >> 2;
  f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int i = slot; i < p.n_part; i += 64) acc += *reinterpret_cast<const f4v*>(p.gain_part + (size_t)i * p.width + col);
  red[tid] = acc;
  __syncthreads();
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) {
    if (slot < s) red[tid] += red[tid + 4 * s];
    __syncthreads();
  }
  if (slot == 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) ((half_t*)p.dgain)[col + e] = (half_t)red[tid][e];
  }
}

hipError_t launch_layer_finish(const LayerFinishParams& p, hipStream_t stream) {
  const int blocks = p.dgain ? p.width / 16 : 0;
  hipLaunchKernelGGL(layer_finish_kernel, dim3(blocks + 1), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace DA_NS
