// Launch parameter blocks of the layer's kernels (layer.hip) and the split of a weight gradient.
#pragma once
#include <hip/hip_runtime.h>
#include "common.hpp"
#include "dispatch.hpp"
#include "layer_abi.h"

namespace da_abi {

// out[E][E] = a^T b over T tokens; a and b are [T][E] with row strides lda and ldb, in the 16-bit type of the build
struct WgradJob {
  const void* a; const void* b;
  void* out;
  int lda, ldb;
};

struct WgradParams {
  WgradJob job[4];
  int n_jobs, T, E;             // E is a multiple of kWgradTile
  WgradSplit split;
  float* part;                  // [splits][n_jobs][E][E], used with more than one split
};

struct LayerPackParams {
  const void* w[3];             // three weights of weight_bytes each (a multiple of 16)
  void* packed;
  size_t weight_bytes;
  diffattn_lambda_vectors vec;
  float* lambda;                // [vec.n]; null: weights only
  float lambda_init;
};

struct LayerFinishParams {
  const float* gain_part;       // [n_part][width]
  int n_part, width;            // width is a multiple of 16
  void* dgain;                  // [width]; null: none wanted
  diffattn_lambda_vectors vec;
  const float* dlambda;         // [vec.n]; null: no vector gradients wanted
  float *dq1, *dk1, *dq2, *dk2;
};

}  // namespace da_abi

namespace da {
hipError_t launch_wgrad(const da_abi::WgradParams& p, hipStream_t stream);
hipError_t launch_layer_pack(const da_abi::LayerPackParams& p, hipStream_t stream);
hipError_t launch_layer_finish(const da_abi::LayerFinishParams& p, hipStream_t stream);
}  // namespace da
namespace da_bf16 {
hipError_t launch_wgrad(const da_abi::WgradParams& p, hipStream_t stream);
hipError_t launch_layer_finish(const da_abi::LayerFinishParams& p, hipStream_t stream);
}  // namespace da_bf16
