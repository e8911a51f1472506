/*
 * What libdiffattn exports for the layer around the operator (modules.DiffAttn), beside the operator's own C ABI
 * (include/diffattn.h): the interface between the library and the layer's extension module (layer_host.cpp).  Conventions
 * and return codes are those of diffattn.h; every pointer is device memory and 16-byte aligned.
 */
#ifndef DIFFATTN_LAYER_ABI_H_
#define DIFFATTN_LAYER_ABI_H_

#include "../../include/diffattn.h"

/* The version of the functions below, raised with every change to their arguments; those of diffattn.h have their own. */
#define DIFFATTN_LAYER_VERSION 2

#ifdef __cplusplus
extern "C" {
#endif

int diffattn_layer_version(void);

/* lambda[o] = exp(q1[o] . k1[o]) - exp(q2[o] . k2[o]) + lambda_init, o < n, vectors of d fp32 values */
typedef struct diffattn_lambda_vectors {
  const float *q1, *k1, *q2, *k2;
  int n, d;
} diffattn_lambda_vectors;

/* Copies three matrices of weight_bytes (a multiple of 16) each one behind the other to `packed` (skipped when weight_bytes
 * is 0; then the matrices and `packed` may be NULL), and forms lambda (skipped when `lambda` is NULL; then `vectors` may be
 * NULL too). */
int diffattn_layer_pack(const void* w0, const void* w1, const void* w2, void* packed, size_t weight_bytes,
                        const diffattn_lambda_vectors* vectors, float lambda_init, float* lambda, void* stream);

/* diffattn_forward_padded without dropout that also, or with y NULL only, writes y * gain (2D values of the tensors' type, one per feature),
 * formed from y as it is stored and rounded once more, to y_gain, in the layout of y. */
int diffattn_layer_forward(const void* q1, const void* q2, const void* k1, const void* k2, const void* v,
                           const void* lambda_scale, void* y, void* u2, float* lse1, float* lse2, float* rinv,
                           int B, int H, int N, int n_valid, int D, float sm_scale, float lambda_init, int flags,
                           const diffattn_layout* layout, const void* gain, void* y_gain, void* stream);

/* diffattn_backward_stages without dropout, with DIFFATTN_RMS_NORM in `flags`, for an output that the caller has multiplied by `gain` (2D values of the tensors' type, one per
 * feature): dy is the gradient of y * gain.  gain_part: diffattn_layer_gain_parts(B, H, N, D) rows of 2D fp32 values, the
 * partial sums of the gain's gradient, written by DIFFATTN_STAGE_PREP. */
size_t diffattn_layer_gain_parts(int B, int H, int N, int D);
int diffattn_layer_backward(const void* q1, const void* q2, const void* k1, const void* k2, const void* v,
                            const void* lambda_scale, const void* y, const void* u2,
                            const float* lse1, const float* lse2, const float* rinv, const void* dy,
                            void* dq1, void* dq2, void* dk1, void* dk2, void* dv, void* dlambda,
                            void* workspace, size_t workspace_bytes,
                            int B, int H, int N, int n_valid, int D, float sm_scale, float lambda_init, int flags,
                            unsigned stage_mask, const diffattn_layout* layout,
                            const void* gain, float* gain_part, void* stream);

/* out[E][E] = a^T b over T tokens, a and b [T][E] with row strides lda and ldb (elements, multiples of 8), for up to four
 * jobs of one size; E is a multiple of 128.  The contraction is split between workgroups where the tiles alone do not fill
 * the chip; workspace: diffattn_layer_wgrad_workspace_bytes (0 when nothing is split).  Bit-reproducible for a
 * given number of jobs; with more or fewer of them the split, and with it the order of a sum, may be another. */
typedef struct diffattn_wgrad_job {
  const void *a, *b;
  void* out;
  long long lda, ldb;
} diffattn_wgrad_job;
size_t diffattn_layer_wgrad_workspace_bytes(int n_jobs, int T, int E);
int diffattn_layer_wgrad(const diffattn_wgrad_job* jobs, int n_jobs, int T, int E, void* workspace, size_t workspace_bytes,
                         int flags /* DIFFATTN_BF16 */, void* stream);

/* dgain[width] = sum of the n_part rows of gain_part (skipped when dgain is NULL), and the gradients of the lambda vectors
 * from dlambda[n] (skipped when it is NULL). */
int diffattn_layer_finish(const float* gain_part, int n_part, int width, void* dgain,
                          const diffattn_lambda_vectors* vectors, const float* dlambda,
                          float* dq1, float* dk1, float* dq2, float* dk2, int flags /* DIFFATTN_BF16 */, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* DIFFATTN_LAYER_ABI_H_ */
