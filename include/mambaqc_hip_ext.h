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

/* fp32 GEMM on the 16-bit matrix cores (each operand split into two fp16 pieces under a
 * power-of-two scale per row, three products per pair of pieces, fp32 accumulation):
 *   Y[m * ldy + n] = sum_k X[m * x_row + k * x_col] * W[n * w_row + k * w_col]
 * for m < M, n < N, k < K. One of x_row and x_col and one of w_row and w_col is 1 (and none
 * is negative), so X and W may be matrices or their transposes: F.linear and both of its
 * gradients (mambaqc/layers/quaternion_linear.py:145-161). Y may not overlap an operand.
 * Accuracy: each element is held to 2^-23 of itself, or to 2^-40 of its row's largest where that
 * is more; outputs that this last may put off by more than 2^-28 K of themselves (2^-20 below
 * K 256), all outputs of rows where more than an eighth of the elements are so small, and of
 * rows with an inf, are computed in plain fp32.
 * workspace: mqc_gemm_f32_workspace_bytes(M, N, K) bytes, 256-byte aligned (MQC_E_SPACE
 * if smaller). */
int64_t mqc_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K);
int mqc_gemm_f32(const float* X, int64_t x_row, int64_t x_col, const float* W, int64_t w_row,
                 int64_t w_col, float* Y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                 void* workspace, int64_t workspace_bytes, void* stream);

/* Up to four small fp32 products in one launch, Y[m * N + n] = sum_k X[m * xm + k * xk] *
 * W[n * wn + k * wk] (+ bias[n]). products: count rows of eleven values, X, xm, xk, W, wn, wk,
 * bias (or 0), Y, M, N, K (pointers as integers; one of xm, xk and one of wn, wk is 1). */
int mqc_gemm_f32_small(const int64_t* products, int64_t count, void* stream);

/* mqc_qln_bwd with its parameter sums: dq, and dgamma [d] and dbeta [d, 4] in fp32. rows and d at
 * least 1, d at most 4096; workspace of mqc_qln_bwd_sums_workspace_bytes(rows, d). */
int64_t mqc_qln_bwd_sums_workspace_bytes(int64_t rows, int64_t d);
int mqc_qln_bwd_sums(const void* q, const void* dout, const float* gamma, const float* mean,
                     const float* rstd, void* dq, float* dgamma, float* dbeta, int64_t rows,
                     int64_t d, float eps, int dtype, void* workspace, int64_t workspace_bytes,
                     void* stream);

/* out_i[c] = sum over r < rows of in_i[r * n_i + c] for up to three fp32 arrays (n_i 0: none),
 * in a fixed order, in one launch. */
int mqc_sum_rows(const float* in1, float* out1, int64_t n1, const float* in2, float* out2,
                 int64_t n2, const float* in3, float* out3, int64_t n3, int64_t rows,
                 void* stream);

/* mqc_cumprod_scan_fwd and mqc_ssm_q_fwd (from a zero state, without h_last) with the sequence
 * in chunks of chunk_len steps walked side by side, for few lanes (batch x lanes, lanes =
 * d_model x d_state for the SSM). chunk_len < seq_len; workspace (16-byte aligned) of
 * mqc_q_chunked_workspace_bytes (ssm 1 for the SSM); batch x chunks at most 65535. */
int64_t mqc_q_chunked_workspace_bytes(int64_t batch, int64_t seq_len, int64_t lanes,
                                      int64_t chunk_len, int ssm);
int mqc_cumprod_scan_chunked(const void* q, void* out, int64_t batch, int64_t seq_len,
                             int64_t lanes, int64_t chunk_len, int dtype, void* workspace,
                             int64_t workspace_bytes, void* stream);
int mqc_ssm_q_fwd_chunked(const void* q, const void* B, const void* Sq, const void* C,
                          const void* D, int64_t d_stride_b, int64_t d_stride_t,
                          int64_t d_stride_d, void* y, int64_t batch, int64_t seq_len,
                          int64_t d_model, int64_t d_state, int64_t chunk_len, int dtype,
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

/* One recurrent decode step of the block in four launches (bf16 or fp16; M = batch, 1 to 16
 * rows, K and 4 d_inner multiples of 32, X within the skinny GEMM's 64 KiB of LDS, else
 * MQC_E_LIMIT). Each rounds to dtype where the separate launches store.
 *
 * mqc_step_in_proj_conv: X [M, K] times W [>= channels + z_cols, K] (+ bias); the first
 * `channels` columns are one step of mqc_causal_conv_silu_step (continued from and shifting
 * tail [M, conv_k - 1, channels]) into act [M, channels], the next z_cols go to z [M, z_cols].
 * channels a multiple of 8, conv_k at most 4.
 * mqc_gemm_skinny4_nt: mqc_gemm_skinny_nt for four weights sharing X.
 * mqc_step_ssm: delta = softplus(dt_raw), s = sigmoid(g_raw) x, then one step of
 * mqc_ssm_fused_fwd in place on h (fp32 [batch, d_inner, d_state, 4]); d_state <= 64.
 * mqc_step_norm_out_gate: mqc_qln_fwd of Y [M, d_inner, 4], times W [d_model, 4 d_inner]
 * (+ bias), out = x + sigmoid(z) * that (x, out [M, d_model]; z rows z_row_stride apart). */
int mqc_step_in_proj_conv(const void* X, int64_t M, int64_t K, const void* W, const void* bias,
                          int64_t channels, int64_t z_cols, const float* conv_w,
                          const float* conv_b, int64_t conv_k, void* tail, void* act, void* z,
                          int dtype, void* stream);
int mqc_gemm_skinny4_nt(const void* X, int64_t M, int64_t K, const void* W1, const void* bias1,
                        void* Y1, int64_t N1, const void* W2, const void* bias2, void* Y2,
                        int64_t N2, const void* W3, const void* bias3, void* Y3, int64_t N3,
                        const void* W4, const void* bias4, void* Y4, int64_t N4, int dtype,
                        void* stream);
int mqc_step_ssm(const void* dt_raw, const void* g_raw, const void* x, const void* B,
                 const void* C, const float* lambda_alpha, const float* lambda_imag,
                 const float* D, float* h, void* y, int64_t batch, int64_t d_inner,
                 int64_t d_state, float eps, int dtype, void* stream);
int mqc_step_norm_out_gate(const void* Y, int64_t M, int64_t d_inner, const float* gamma,
                           const float* beta, float eps, const void* W, const void* bias,
                           int64_t d_model, const void* x, const void* z, int64_t z_row_stride,
                           void* out, int dtype, void* stream);
/* 1 where mqc_step_norm_out_gate takes M rows of d_inner quaternions, else 0. */
int mqc_step_norm_out_gate_fits(int64_t M, int64_t d_inner);

#ifdef __cplusplus
}
#endif

#endif /* MAMBAQC_HIP_EXT_H */
