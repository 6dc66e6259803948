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

/* Linear layers of many rows that share their input, as one launch (bf16): out[i]
 * [M,N[i]] = x [M,K] . w[i] [N[i],K]^T + bias[i] (bias or an entry of it NULL: none), and
 * the stacked layer of the MLP with its join, out [M,N] = gelu(x . w[0] + bias[0]) *
 * (x . w[1] + bias[1]) with w [2,K,N], bias [2,N] or NULL.  Float32 sums, each product
 * rounded once; K a multiple of 64, N of 8, else RG_ERR_UNSUPPORTED.  *_pays: whether
 * that is ahead of the library's products. */
int rg_linear_many_pays(int64_t M, int K, int count, const int* N, int dtype);
int rg_linear_many(const void* x, int64_t M, int K, int count, const void* const* w,
                   const void* const* bias, void* const* out, const int* N, int dtype,
                   void* stream);
int rg_linear_gelu_pair_pays(int64_t M, int K, int N, int dtype);
int rg_linear_gelu_pair(const void* x, const void* w, const void* bias, void* out,
                        int64_t M, int K, int N, int dtype, void* stream);

/* rg_linear_many, rg_linear_gelu_pair and rg_add_rms_norm (bf16) of some of the rows of
 * tensors with `rows` of them: those in `count` runs of eight, which start at the rows in
 * `runs` (on the GPU, 0 .. rows - 8, any order, overlaps allowed); nothing else is read or
 * written.  RG_ERR_UNSUPPORTED beyond the sizes of those calls (norm: rows of at most 4096
 * in eights).  *_serve: whether tensors of `rows` rows are within them: (rows + 512) times
 * the widest of K and N below 2^30, however few rows the runs have.  *_saves_us: what
 * `count` runs take less than all rows as they are run better, here or by the library, by
 * the times that their rules go by (below zero: they take more). */
int rg_linear_many_runs_serve(int64_t rows, int K, int layers, const int* N, int dtype);
int rg_linear_gelu_pair_runs_serve(int64_t rows, int K, int N, int dtype);
double rg_linear_many_runs_saves_us(int64_t rows, int count, int K, int layers,
                                    const int* N, int dtype);
double rg_linear_gelu_pair_runs_saves_us(int64_t rows, int count, int K, int N, int dtype);
int rg_linear_many_runs(const void* x, int64_t rows, const int32_t* runs, int count, int K,
                        int layers, const void* const* w, const void* const* bias,
                        void* const* out, const int* N, int dtype, void* stream);
int rg_linear_gelu_pair_runs(const void* x, const void* w, const void* bias, void* out,
                             int64_t rows, const int32_t* runs, int count, int K, int N,
                             int dtype, void* stream);
int rg_add_rms_norm_runs(const void* x, const void* addend, const void* scale,
                         void* sum_out, void* out, const int32_t* runs, int count,
                         int width, float eps, int dtype, void* stream);

/* What such layers give back: dx [M,N] = dy [M,K] . w [K,N] (+ dy2 . w2 of the same
 * sizes: two layers that read the same x; both NULL: none), one rounding; and dw[i]
 * [out_features[i], in_features[i]] = dy[i] [M,out]^T . x[i] [M,in], up to four as one
 * launch (features in multiples of 8, any M).  The latter has no rule of its own: its
 * contraction fills the tiles whatever the rows (library / this, us: three of 2560 x 2560
 * over 256 rows 60 / 21, 1000 rows 87 / 37, 8192 rows 407 / 211, one of 4096 x 4096 over
 * 8192 rows 237 / 181; of widths 64 to 4096, 70 to 32768 rows and one to three layers
 * behind by more than 2 us only with 4096 x 4096 over 70 to 300 rows, 17 / 20 and three
 * of them 69 / 75, and one of 256 x 256 over 32768 rows, 114 / 126). */
int rg_linear_back_pays(int64_t M, int K, int N, int two, int dtype);
int rg_linear_back(const void* dy, const void* w, const void* dy2, const void* w2,
                   void* dx, int64_t M, int K, int N, int dtype, void* stream);
int rg_linear_weight_grads(const void* const* dy, const void* const* x, void* const* dw,
                           const int* out_features, const int* in_features, int count,
                           int64_t M, int dtype, void* stream);

/* rg_linear_rows without a residual, and bytes (a multiple of 16) copied from `from` to
 * `to` beside it: a state that the next launch on the stream reads from the copy while it
 * overwrites the original.  RG_ERR_UNSUPPORTED where rg_linear_rows wants a workspace. */
int rg_linear_rows_beside(const void* x, const void* w_packed, const void* bias, void* out,
                          int M, int K, int N, int groups, const void* from, void* to,
                          int64_t bytes, void* stream);

/* rg_recurrent_step and rg_gelu_mul of its y with gate_branch [B,1,W], one launch where
 * the step is one (float32, 256-wide heads, nothing written that is read). */
int rg_recurrent_step_join(const void* x, const void* gate_branch, const void* segpos,
                           int segpos_is_i64, const void* conv_cache_in,
                           void* conv_cache_out, const void* h_in, void* h_out,
                           const void* conv_w, const void* conv_b, const void* w_x,
                           const void* b_x, const void* w_a, const void* b_a,
                           const void* a_param, void* y, void* workspace,
                           size_t workspace_bytes, int B, int W, int H, int dtype,
                           void* stream);

/* rg_linear_rows_partial that also sets the RG_NORM_FLAGS words of `flags` to zero, for
 * rg_linear_rows_normed: rg_add_rms_norm_partial of such sums (M rows of K; sum_out and
 * normed are written whole) and rg_linear_rows of normed, without a residual, as one
 * launch, with `bytes` copied as in rg_linear_rows_beside (0: none).  The flags serve one
 * such launch.  patience: how often its workgroups look for the rows' norm before they
 * form it themselves.  out has the same bits as the two calls.  RG_ERR_UNSUPPORTED where *_serve says 0. */
#define RG_NORM_FLAGS 64
int rg_linear_rows_partial_flags(const void* x, const void* w_packed, void* partial,
                                 uint32_t* flags, int M, int K, int N, int slices,
                                 void* stream);
int rg_linear_rows_normed_serve(int M, int K, int N, int gelu_pair);
int rg_linear_rows_normed(const void* partial, int slices, const void* partial_bias,
                          const void* addend, const void* scale, float eps, void* sum_out,
                          void* normed, uint32_t* flags, const void* w_packed,
                          const void* bias, void* out, int M, int K, int N, int groups,
                          int gelu_pair, const void* from, void* to, int64_t bytes,
                          int patience, void* stream);

#ifdef __cplusplus
}
#endif

#endif  /* RG_PACKAGE_CALLS_H_ */
