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

#ifdef __cplusplus
}
#endif
