/* Entry points of libmambaqc_hip.so beside the drop-in boundary of mambaqc_hip.h: products
 * and fused steps that the Python layers choose by size, each computing what operators of
 * mambaqc_hip.h or torch compute otherwise. Conventions, status codes and dtype codes are
 * that header's. */
#ifndef MAMBAQC_HIP_EXT_H
#define MAMBAQC_HIP_EXT_H

#include "mambaqc_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* fp32 GEMM at fp32 accuracy on the 16-bit matrix cores (each operand split into two fp16
 * pieces under a power-of-two scale per row, three products per pair of pieces, fp32
 * accumulation; rows with an inf or a NaN are computed in plain fp32):
 *   Y[m * ldy + n] = sum_k X[m * x_row + k * x_col] * W[n * w_row + k * w_col]
 * for m < M, n < N, k < K. One of x_row and x_col and one of w_row and w_col is 1 (and none
 * is negative), so X and W may be matrices or their transposes: F.linear and both of its
 * gradients (mambaqc/layers/quaternion_linear.py:145-161). Y may not overlap an operand.
 * workspace: mqc_gemm_f32_workspace_bytes(M, N, K) bytes, 256-byte aligned (MQC_E_SPACE
 * if smaller). */
int64_t mqc_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K);
int mqc_gemm_f32(const float* X, int64_t x_row, int64_t x_col, const float* W, int64_t w_row,
                 int64_t w_col, float* Y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                 void* workspace, int64_t workspace_bytes, void* stream);

/* mqc_ssm_fused_bc_fwd for short sequences, seq_len from 1 to 128 (MQC_E_LIMIT above): same
 * operands, dtypes, shapes and refusals, in tiles of 64 or 128 tokens that hold whole
 * sequences of the batch, each group of 16 states in a workgroup of its own. d_state > 16
 * needs workspace (mqc_ssm_fused_bc_short_workspace_bytes, 16-byte aligned) for the groups'
 * partial sums of y. h_last may be h0. */
int64_t mqc_ssm_fused_bc_short_workspace_bytes(int64_t batch, int64_t seq_len, int64_t d_inner,
                                               int64_t d_state);
int mqc_ssm_fused_bc_short_fwd(const void* x, const void* B_weight, const void* C_weight,
                               const void* delta, const void* s, const float* lambda_alpha,
                               const float* lambda_imag, const float* D, const void* h0, void* y,
                               void* h_last, int64_t batch, int64_t seq_len, int64_t d_inner,
                               int64_t d_state, float eps, int dtype, void* workspace,
                               int64_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MAMBAQC_HIP_EXT_H */
