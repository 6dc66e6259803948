/* Entry points that this package's own Python calls beside the public C
 * interface of include/rg_lru.h (same conventions: device pointers, a stream,
 * RG_OK or an error code, rg_last_error): steps fused the way its modules chain
 * them, free to change with those. */
#ifndef RG_PACKAGE_CALLS_H_
#define RG_PACKAGE_CALLS_H_

#include "../../include/rg_lru.h"

#ifdef __cplusplus
extern "C" {
#endif

/* first_key of rg_attention_prefill for a prompt's positions [B,T]
 * (int32/int64): max(last position 0 at or before the query, else 0;
 * t - window) -- the mask of recurrentgemma/torch/modules.py:86-127. */
int rg_attention_first_key(const void* positions, int positions_is_i64,
                           int32_t* first_key, int B, int T, int window,
                           void* stream);

/* A prompt pass of the local-attention block between its projections
 * (modules.py:431-476, ring cache :253-283) in two launches: rg_rope_pair on q
 * and k, rg_attention_prefill, and the cache it leaves.  q, out [B,T,H,256],
 * k, v [B,T,256] as the projections leave them, inv_freq [64], first_key
 * [B,T]; ring_keys, ring_values [B,window,256] and num_tokens [B] are written
 * whole (all three NULL: no cache); workspace of
 * rg_attention_prompt_workspace_bytes(B, T).  RG_ERR_UNSUPPORTED as for
 * rg_attention_prefill. */
size_t rg_attention_prompt_workspace_bytes(int B, int T);
int rg_attention_prompt(const void* q, const void* k, const void* v,
                        const void* positions, int positions_is_i64,
                        const float* inv_freq, const int32_t* first_key,
                        void* out, void* ring_keys, void* ring_values,
                        int32_t* num_tokens, void* workspace, int B, int T,
                        int H, int head_dim, int window, float scale, int dtype,
                        void* stream);

/* rg_argmax_rows with several workgroups to a row, which need a workspace of
 * rg_argmax_workspace_bytes (0: one workgroup is enough, and workspace may be
 * NULL). */
size_t rg_argmax_workspace_bytes(int rows, int n);
int rg_argmax_rows_split(const void* x, int64_t* out, void* workspace, int rows,
                         int n, int dtype, void* stream);

/* The workspace with which rg_recurrent_core is fastest: what it needs or, where a
 * form with a larger one is ahead (float32 shapes that one launch serves as well, bf16
 * rows that come out uneven on the CUs), what that takes. */
size_t rg_recurrent_core_best_workspace_bytes(int B, int T, int W, int H,
                                              int dtype);

/* The bare recurrence with the workspace that it is fastest with, forward by
 * rg_linear_scan_split and backward by rg_linear_scan_backward_best (0: none). */
size_t rg_linear_scan_best_workspace_bytes(int B, int T, int W, int dtype,
                                           int backward);
int rg_linear_scan_backward_best(const void* dy, const void* a, const void* reset,
                                 const void* y, const void* h0, const void* dh_last,
                                 void* dx, void* da, void* dh0, void* workspace,
                                 size_t workspace_bytes, int B, int T, int W,
                                 int dtype, void* stream);

/* Bytes with which a recurrence's one-pass kernel is dealt out in steps, 0 where it is
 * not: mode 0 the plain forward, 1 the plain backward, 2 and 3 the gated ones. */
size_t rg_scan_deal_bytes(int B, int T, int W, int dtype, int mode);

#ifdef __cplusplus
}
#endif

#endif  /* RG_PACKAGE_CALLS_H_ */
