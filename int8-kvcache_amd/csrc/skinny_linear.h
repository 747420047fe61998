/*
 * skinny_linear.h -- the decode step's matrix products (a few activation rows times a large bf16
 * weight matrix), exported by libint8kv.so for the package's own decode loop.  Not part of the
 * public C ABI (include/): the entry points may change with the loop that calls them.
 *
 * Conventions are those of include/int8kv.h: device pointers, element strides, a hipStream_t as
 * void*, 0 / negative INT8KV_E_* / positive hipError_t returns, no allocation, no
 * synchronisation.  Every matrix is bf16 with 16-byte aligned rows and a unit inner stride.
 */
#ifndef INT8KV_SKINNY_LINEAR_H
#define INT8KV_SKINNY_LINEAR_H

#include <stdint.h>

#include "../../include/int8kv.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Whether the products below take x [rows, k] times w [n, k]^T (else INT8KV_E_SHAPE):
 * 1 <= rows <= 32, k a positive multiple of 64 up to 32768,
 * n a positive multiple of 16. */
int32_t int8kv_skinny_linear_ok(int64_t rows, int64_t k, int64_t n);

/* Workspace of int8kv_skinny_linear_add_rms_norm (fp32 partial sums; no initialisation needed). */
int64_t int8kv_skinny_linear_workspace_bytes(int64_t rows, int64_t k, int64_t n);

/* out[r, j] = bf16(sum_i x[r, i] w[j, i] + bias[j]) with fp32 products and sums; bias may be
 * NULL.  workspace as above (used when k is split over workgroups). */
int int8kv_skinny_linear(const void* x, int64_t rows, int64_t k, int64_t x_row_stride,
                         const void* w, int64_t n, int64_t w_row_stride, const void* bias,
                         void* out, int64_t out_row_stride, void* workspace,
                         int64_t workspace_bytes, void* stream);

/* out[r, j] = bf16(bf16(silu(g)) u) with g = bf16(x w[j]^T), u = bf16(x w[ffn + j]^T):
 * int8kv_skinny_linear by w [2 ffn, k] followed by int8kv_silu_mul.  k: at most 4096; ffn: a
 * multiple of 8. */
int int8kv_skinny_linear_silu_mul(const void* x, int64_t rows, int64_t k, int64_t x_row_stride,
                                  const void* w, int64_t ffn, int64_t w_row_stride, void* out,
                                  int64_t out_row_stride, void* stream);

/* residual[r, :] = bf16(residual[r, :] + bf16(x w^T)[r, :]) and the RMSNorm of it into `out`:
 * int8kv_skinny_linear by w [n, k] followed by int8kv_add_rms_norm (n = hidden, at most 8192). */
int int8kv_skinny_linear_add_rms_norm(const void* x, int64_t rows, int64_t k,
                                      int64_t x_row_stride, const void* w, int64_t n,
                                      int64_t w_row_stride, void* residual,
                                      int64_t residual_row_stride, const void* norm_weight,
                                      void* out, int64_t out_row_stride, float eps,
                                      void* workspace, int64_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* INT8KV_SKINNY_LINEAR_H */
