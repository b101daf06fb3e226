// Entry points of libmce.so for this package's own Python layer, beside the
// public C ABI of mce_abi.h (same conventions: raw device pointers, element
// counts and strides, a hipStream_t passed as void *, an MCE_* status).
#pragma once

#include "mce_abi.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * mce_prefill_attention over strided q, k and v: element strides between
 * sequences and between positions (rows of all heads are contiguous, heads 128
 * apart; k and v share theirs), multiples of 8.  The engine passes views into
 * the fused q/k/v projection output.  out is contiguous.
 */
MCE_API int mce_prefill_attention_strided(int dtype, const void *query, const void *key,
                                          const void *value, void *output, int batch, int seq_len,
                                          int num_heads, int num_kv_heads, int head_dim,
                                          int64_t q_seq_stride, int64_t q_row_stride,
                                          int64_t kv_seq_stride, int64_t kv_row_stride,
                                          float scale, void *stream);

/*
 * A projection of a prompt: out[m, n] (op)= x[m, k] . w[n, k]^T ([2 n, k] gate
 * rows then up rows for SwiGLU), epilogues as mce_decode_gemm; with the residual
 * add and a norm weight, also normed[m, n] = RMSNorm(out) (mce_rmsnorm's bits
 * for the updated rows).  Takes the sizes at which it is faster than the
 * library GEMM and answers MCE_ERR_UNSUPPORTED, with nothing done, to all
 * others.  Needs mce_prompt_gemm_workspace_size() bytes, 256-byte aligned (0: a
 * null pointer is fine; no initialisation; calls that run concurrently need
 * their own).  x_stride / out_stride: elements between rows, multiples of 8.
 */
MCE_API int mce_prompt_gemm_takes(int m, int n, int k, int epilogue);  /* 1: takes the sizes */
MCE_API size_t mce_prompt_gemm_workspace_size(int m, int n, int k, int epilogue);
MCE_API int mce_prompt_gemm(int dtype, const void *x, const void *w, void *out, int m, int n, int k,
                            int64_t x_stride, int64_t out_stride, int epilogue,
                            const void *norm_weight, float eps, void *normed, void *workspace,
                            size_t workspace_bytes, void *stream);

#ifdef __cplusplus
}
#endif
