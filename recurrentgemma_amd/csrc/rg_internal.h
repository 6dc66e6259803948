// Launcher declarations shared by the kernel files and the C-ABI file.
#ifndef RG_INTERNAL_H_
#define RG_INTERNAL_H_

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

namespace rg {

// How document starts are encoded: int32 / int64 positions (start == 0), or a
// byte mask (start != 0) as rnn_scan's `reset` argument.
enum SegKind { kSegI32 = 0, kSegI64 = 1, kSegMaskU8 = 2 };

// Raises a kernel's dynamic LDS limit the first time it is launched on a
// device; later launches on that device only read the flag (the attribute is a
// property of the loaded function, it does not have to be set per launch).
struct OncePerDevice {
  std::atomic<uint64_t> done{0};  // bit d: set on device d (d < 64)
};
inline hipError_t set_max_dynamic_lds(OncePerDevice& once, const void* fn,
                                      size_t bytes) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (dev < 64 && (once.done.load(std::memory_order_acquire) & bit))
    return hipSuccess;
  e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)bytes);
  if (e == hipSuccess && dev < 64)
    once.done.fetch_or(bit, std::memory_order_release);
  return e;
}

struct ConvArgs {
  const void* x;
  const void* segpos;
  int seg_kind;  // 0: int32 positions, 1: int64 positions, 2: byte mask
  const void* w;
  const void* bias;
  void* out;
  void* cache_out;
  int B, T, W, K;
};

struct ConvStepArgs {
  const void* x;
  const void* cache_in;
  const void* w;
  const void* bias;
  void* out;
  void* cache_out;
  int B, W, K;
};

struct GemmArgs {
  const void* x;       // [M, W]
  int apply_conv;      // width-4 conv on load
  const void* segpos;  // [M] (only with apply_conv)
  int seg_kind;
  const void* conv_w;  // [4, W]
  const void* conv_b;  // [W]
  const void* w[2];    // [H, bw, bw] per gate
  const void* b[2];    // [H, bw] per gate
  void* out[2];        // [M, W] per gate
  int ngates;          // 1 or 2
  int64_t M;           // rows = B*T
  int T;               // sequence length (row m is token m % T of its row)
  int W, H, bw;
};

struct ScanArgs {
  int plain;  // 1: rnn_scan only (x is the recurrence input, ga holds a)
  const void* x;
  int apply_conv;
  const void* conv_w;
  const void* conv_b;
  const void* gx;
  const void* ga;
  const void* a_param;
  const void* segpos;
  int seg_kind;
  const float* h0;
  void* y;
  float* h_last;
  void* cache_out;
  int B, T, W;
  // sequences cut into `chunks` chunks of t_chunk tokens (chunks <= 1: not
  // cut), with three [B][chunks][W] float rows of workspace: every chunk's
  // product of a_t, its state from a zero start, its incoming state
  int chunks, t_chunk;
  float* ws_p;
  float* ws_h;
  void* deal;  // plain: as in ScanTileArgs
};

struct FusedArgs {
  const void* x;       // [B, T, W] bf16, the conv input
  const void* segpos;  // [B, T]
  int seg_kind;
  const void* conv_w;  // [4, W]
  const void* conv_b;  // [W]
  const void* w[2];    // [H, 256, 256]: input gate, a gate
  const void* w_packed;  // or null: both, see launch_pack_gate_weights
  const void* b[2];    // [H, 256]
  const void* a_param; // [W]
  const float* h0;     // [B, W] or null
  void* y;             // [B, T, W]
  // or null: [B, T, W] bf16, the other branch of the recurrent block before
  // its activation; y is then the block's join y * gelu(gate_branch)
  const void* gate_branch;
  float* h_last;       // [B, W] or null
  void* cache_out;     // [B, 3, W] or null
  int B, T, W, H;
  // sequences cut into `chunks` chunks of tiles_per_chunk 64-token tiles
  // (chunks <= 1: not cut), with two [B][chunks][W] float rows of workspace:
  // every chunk's product of a_t and its state from a zero start
  int chunks, tiles_per_chunk;
  float* ws_p;
  float* ws_h;
  // rg_prefill_relay.hip: states between blocks, tickets taken per head
  uint64_t* relay_words;
  int* relay_tickets;
  // or null: workgroup (0, 0) leaves here the shader-clock cycles and the
  // 100 MHz ticks its tile loop took (rg_prefill_clock_probe)
  uint64_t* timing;
};

struct StepArgs {
  const void* x;         // [B, 1, W] bf16
  const void* segpos;    // [B, 1]
  int seg_kind;
  const void* cache_in;  // [B, 3, W] bf16
  void* cache_out;       // [B, 3, W] bf16 (may alias cache_in)
  const float* h_in;     // [B, W]
  float* h_out;          // [B, W] (may alias h_in)
  const void* conv_w;
  const void* conv_b;
  const void* w_packed;  // both gate matrices, see launch_pack_gate_weights
  const void* b[2];
  const void* a_param;
  void* y;               // [B, 1, W]
  // the block's other branch [B, 1, W] or null: y is written as
  // y * gelu(gate_branch)
  const void* gate_branch;
  int B, W, H;
};

// The float32 step in one launch (rg_step_f32.hip): as StepArgs, weights [H, 256, 256].
struct StepF32Args {
  const float* x;
  const void* segpos;
  int seg_kind;
  const float* cache_in;
  float* cache_out;
  const float* h_in;
  float* h_out;
  const float* conv_w;
  const float* conv_b;
  const float* w[2];
  const float* b[2];
  const float* a_param;
  float* y;
  const float* gate_branch;
  int B, W, H;
};

// Prompt-pass attention (rg_attention_prefill.hip).
struct AttnPrefillArgs {
  const void* q;    // [B, T, H, 256] bf16, after the rotary embedding
                    // (before it where rope_table is given)
  const void* k;    // [B, T, 256] bf16, after the rotary embedding
  const void* v;    // [B, T, 256] bf16, or (T_pad > 0) [B, 256, T_pad]: transposed, zeros
                    // behind token T - 1 (T_pad a multiple of 64)
  const void* lo;   // [B, T] int32: first key each query sees (non-decreasing)
  void* out;        // [B, T, H, 256] bf16
  int B, T, T_pad, H;
  float scale;      // of the scores (head_dim ** -0.5)
  const uint32_t* rope_table;  // [B, T, 64] (sine, cosine) pairs, or null
};
hipError_t launch_attn_prefill_bf16(const AttnPrefillArgs& a, hipStream_t s);
// What precedes it in a block (same file).
struct AttnPromptArgs {
  const uint16_t* k;      // [B, T, 256] before the rotary embedding
  const uint16_t* v;      // [B, T, 256]
  const void* pos;        // [B, T]
  int pos_kind;
  const float* inv_freq;  // [64]
  uint16_t* k_rot;        // [B, T, 256]
  uint32_t* rope_table;   // [B, T, 64]
  uint16_t* ring_k;       // [B, window, 256], null: no cache wanted
  uint16_t* ring_v;
  int32_t* num_tokens;    // [B]
  int B, T, window;
  unsigned groups;        // workgroups per row (set by the launch)
};
hipError_t launch_attn_prompt_prepare(const AttnPromptArgs& a, hipStream_t s);
hipError_t launch_first_key(const void* pos, int pos_kind, int32_t* first,
                            int B, int T, int window, hipStream_t s);

// One decoded token against the ring cache (rg_attention_decode.hip).
constexpr int kAttnDecodeChunk = 256;     // ring slots per workgroup
constexpr int kAttnDecodeMaxChunks = 64;  // window <= 16384
struct AttnDecodeArgs {
  const uint16_t* q;      // [B, heads, 256] rows ldq apart, before the rotary
  const uint16_t* k_new;  // [B, 256] rows ldk apart, before the rotary
  const uint16_t* v_new;  // [B, 256] rows ldv apart
  int64_t ldq, ldk, ldv;  // in elements
  const void* pos;        // [B] positions of the new tokens
  int pos_kind;           // 0: int32, 1: int64
  const float* inv_freq;  // [64]
  uint16_t* ring_k;       // [B, window, 256]
  uint16_t* ring_v;
  int32_t* num_tokens;    // [B] tokens seen before this one
  uint16_t* out;          // [B, heads, 256]
  float* part_o;          // [B, chunks, heads, 256]
  float* part_ml;         // [B, chunks, heads, 2]: maximum, denominator
  int B, heads, window, chunks;
  float scale;
  int update;             // write the ring slot and count the token
};
hipError_t launch_attn_decode_fused(const AttnDecodeArgs& a, hipStream_t s);

struct LinearArgs {
  const void* x;         // [M, K] bf16
  const void* w_packed;  // see launch_linear_pack
  const void* bias;      // [N] or null
  const void* residual;  // laid out like out, or null
  void* out;             // [G, M, N / G]; gelu pairs: [M, N / 2]
  float* partial;        // [slices, M, N] when K is split over the grid
  int M, K, N;
  int group_width;       // N / G
  // launch_linear_rows_beside: 16-byte items that workgroups behind the layer's copy
  const void* copy_from;
  void* copy_to;
  int64_t copy_items;
  // with partial sums: kNormFlags words set to zero for launch_linear_rows_normed
  uint32_t* clear;
};
constexpr int kNormFlags = 64;

// A layer whose x is the norm of what the layer before left as partial sums.
struct NormedLinearArgs {
  LinearArgs layer;  // x = normed
  const float* sums;  // [slices, M, K]
  const void* bias;   // [K] or null: of the layer before
  const void* addend;  // [M, K] or null
  const void* scale;   // [K]
  void* sum_out;       // [M, K]
  void* normed;        // [M, K]
  uint32_t* flags;     // kNormFlags words, zero: row m is there
  int slices, patience;
  float eps;
};

// Each returns hipSuccess or the launch error.  dtype: 0 = f32, 1 = bf16.
hipError_t launch_conv1d_prefill(const ConvArgs& a, int dtype, hipStream_t s);
hipError_t launch_conv1d_step(const ConvStepArgs& a, int dtype, hipStream_t s);
struct ConvBwdArgs {
  const void* dout;  // [B, T, W] gradient of the conv output
  const void* x;     // [B, T, W] the conv input
  const void* segpos;
  int seg_kind;
  const void* w;     // [K, W]
  void* dx;          // [B, T, W]
  float* partial;    // [conv1d_backward_chunks(B, T)][K + 1][W]
  float* dx_sums;    // or null: [chunks][W], each chunk's column sums of dx (only
                     // where conv1d_backward_sums_dx)
  int B, T, W, K;
};
int conv1d_backward_chunks(int B, int T);
bool conv1d_backward_sums_dx(int B, int T, int W, int K, int dtype);
hipError_t launch_conv1d_backward(const ConvBwdArgs& a, int dtype,
                                  hipStream_t s);
hipError_t launch_gemm_generic(const GemmArgs& a, int dtype, hipStream_t s);
hipError_t launch_gemm_mfma_bf16(const GemmArgs& a, hipStream_t s);
hipError_t launch_gemm_mfma_f32(const GemmArgs& a, hipStream_t s);
hipError_t launch_lru_scan(const ScanArgs& a, int dtype, hipStream_t s);

// Linear layers of many rows, bf16 (rg_matmul.hip): up to kMaxMatmuls products of one
// kind as one launch.
enum MatmulKind {
  kMatmulForward = 0,   // m [M, K], n [N, K]: c = m n^T + bias
  kMatmulBack = 1,      // m [M, K], n [K, N]: c = m n (+ m2 n2, the same sizes)
  kMatmulWeights = 2,   // m [K, M], n [K, N]: c = m^T n
  kMatmulGeluPair = 3   // m [M, K], n, n2 [K, N]: c = gelu(m n + bias) * (m n2 + bias2)
};
constexpr int kMaxMatmuls = 4;
struct MatmulProblem {
  const void *m, *n, *m2, *n2, *bias, *bias2;
  void* c;                 // [M, N]
  int M, N, K;
  int ldm, ldn, ldc;       // elements from one row of a tensor to the next
  int first_tile;          // (the launcher's)
};
struct MatmulArgs {
  MatmulProblem p[kMaxMatmuls];
  int count;
  // or null: of the tensors' `rows` rows only those in runs of eight, which start at
  // these; p[].M is eight times their number (forward and pairs, any order, runs may
  // overlap)
  const int* runs;
  int rows;
};
// Whether the launch can be made; and (but for weight gradients) whether it is ahead of
// the library's products.
bool matmul_serves(const MatmulArgs& a, int kind);
float matmul_us(const MatmulArgs& a, int kind);
bool matmul_pays(const MatmulArgs& a, int kind);
hipError_t launch_matmul(MatmulArgs a, int kind, hipStream_t s);

// Backward pass of rnn_scan (rg_scan_bwd.hip).
struct ScanBwdArgs {
  const void* dy;        // [B, T, W] gradient of y
  const void* a;         // [B, T, W] the forward coefficients
  const void* reset;     // [B, T] bytes
  const void* y;         // [B, T, W] the forward outputs
  const float* h0;       // [B, W] or null
  const float* dh_last;  // [B, W] or null: gradient of the final state
  void* dx;              // [B, T, W]
  void* da;              // [B, T, W]
  float* dh0;            // [B, W] or null
  int B, T, W;
  void* deal;            // as in ScanTileArgs
};
hipError_t launch_linear_scan_backward(const ScanBwdArgs& a, int dtype,
                                       hipStream_t s);
struct RglruBwdArgs {
  const void* dy;        // [B, T, W] gradient of y
  const void* x;         // [B, T, W] the RG-LRU's input (the conv output)
  const void* gx;        // [B, T, W] input gate pre-activations
  const void* ga;        // [B, T, W] recurrence gate pre-activations
  const void* a_param;   // [W]
  const void* reset;     // [B, T] bytes
  const void* y;         // [B, T, W] the forward outputs
  const float* h0;       // [B, W] or null
  const float* dh_last;  // [B, W] or null: gradient of the final state
  void* dx;              // [B, T, W]
  void* dgx;             // [B, T, W]
  void* dga;             // [B, T, W]
  float* dlam;           // [B, W]: each row's share of a_param's gradient
  float* dh0;            // [B, W] or null
  int B, T, W;
};
hipError_t launch_rglru_backward(const RglruBwdArgs& a, int dtype,
                                 hipStream_t s);
// One pass over every element, 16 bytes of channels per lane
// (rg_scan_tiles.hip).
struct ScanTileArgs {
  // forward: x, a | gated: x, input gate, recurrence gate (pre-activations),
  // float32: the other branch or null
  // backward: dy, a, y | gated: dy, x, input gate, recurrence gate, y
  const void* in[5];
  const void* flags;     // [B, T] document starts
  int flag_kind;         // SegKind
  const void* a_param;   // [W], gated
  const void* bias[2];   // gated float32: [W] or null, added to the input and
                         // recurrence gates' pre-activations
  const float* init;     // [B, W] or null: h0 | backward: dh_last
  const float* h0;       // backward: [B, W] or null
  void* out[3];          // y | dx, da | dx, d input gate, d recurrence gate
  float* last;           // [B, W] or null: h_last | dh0
  float* dlam;           // [B, W], gated backward: each row's share
  float* dbias;          // gated float32 backward, or null: [2][B, W], each
                         // row's sums of the gates' gradients
  // gated forward, or null: what the backward pass is to read in place of
  // tensors that the caller may have written to by then
  uint8_t* starts_out;   // [B, T], 1 where a document starts
  float* bias_out;       // float32: [2][W]
  int B, T, W;
  // or null: scan_tiles_deal_bytes of workspace (16-byte aligned), and the steps of
  // all rows are dealt out to one workgroup per CU; dlam and dbias are then
  // [B * scan_tiles_steps, W] and [2][B * scan_tiles_steps, W], a row per step
  void* deal;
};
// what it takes; 0 where a slab by the workgroup is the faster form
size_t scan_tiles_deal_bytes(int B, int T, int W, int dtype, int mode);
int scan_tiles_steps(int T, int mode);
enum ScanTileMode { kTilesFwdPlain, kTilesBwdPlain, kTilesFwdGated, kTilesBwdGated,
                    // (a question only) both gated ones of a float32 RG-LRU
                    kTilesPairGated };
// whether it takes the shape; ... and is the faster form for it
bool scan_tiles_take(int T, int W, int dtype);
bool scan_tiles_serve(int B, int T, int W, int dtype, int mode);
// whether rg_scan_bwd.hip's kernels give a lane two channels (else one)
bool scan_backward_two_channels(int B, int W);
hipError_t launch_scan_tiles(const ScanTileArgs& a, int mode, int dtype,
                             hipStream_t s);
void scan_split_plan(int B, int T, int W, int granule, int* chunks,
                     int* t_chunk);
// Chunk lengths are multiples of this for the kernel that handles (dtype, W).
int scan_split_granule(int dtype, int W);
hipError_t launch_block_prefill_bf16(const FusedArgs& a, hipStream_t s);
hipError_t launch_block_prefill_teams_bf16(const FusedArgs& a, hipStream_t s);
// the same with blocks of 32 tokens dealt out and states handed on in memory
bool prefill_relay_pays(int B, int H, int T, bool joined);
size_t prefill_relay_workspace_bytes(int B, int W, int H);
hipError_t launch_block_prefill_relay_bf16(FusedArgs a, void* workspace,
                                           hipStream_t s);
// the same for heads of 128 .. 256 channels, cut into slices of 64: few (row,
// head) pairs, short rows, narrower heads (rg_prefill_slices.hip)
bool prefill_short_serves(int B, int H, int T);  // 256-wide heads
hipError_t launch_block_prefill_short_bf16(const FusedArgs& a, hipStream_t s);
bool prefill_slices_serve(int B, int H, int T, bool joined);  // 256-wide heads
// rows of a few tokens, several to a tile (with re-laid-out weights)
bool prefill_many_serve(int B, int H, int T, int bw, bool joined, bool conv, bool state);
bool prefill_narrow_pays(int B, int H, int T, int W);         // narrower ones
hipError_t launch_block_prefill_slices_bf16(const FusedArgs& a, hipStream_t s);
// float32, 256-wide heads, few rows: conv, gate projections, gates and
// recurrence in one launch (rg_core_f32.hip)
bool core_f32_small_serves(int B, int T, int W, int H);
hipError_t launch_core_f32_small(const FusedArgs& a, hipStream_t s);
void prefill_chunk_plan(int B, int H, int T, int* chunks, int* tiles_per_chunk);
hipError_t launch_block_step_bf16(const StepArgs& a, hipStream_t s);
// out[i] = a[i] * gelu_tanh(g[i]) over n elements (out may alias a or g).
hipError_t launch_gelu_mul(const void* a, const void* g, void* out, int64_t n,
                           int dtype, hipStream_t s);
hipError_t launch_gelu_mul_backward(const void* dout, const void* a,
                                    const void* g, void* d_a, void* d_g,
                                    int64_t n, int dtype, hipStream_t s);
// out = tanh(x / cap) * cap, n elements; out[r] = argmax(x[r, :n])
hipError_t launch_soft_cap(const void* x, void* out, int64_t n, float cap,
                           int dtype, hipStream_t s);
size_t argmax_workspace_bytes(int rows, int n);
// workspace: null, or of argmax_workspace_bytes (a row by several workgroups)
hipError_t launch_argmax_rows(const void* x, int64_t* out, void* workspace,
                              int rows, int n, int dtype, hipStream_t s);
// out[r, :] = v * rsqrt(mean(v^2) + eps) * (scale + 1) with v = x[r, :], or,
// with an addend, v = x[r, :] + addend[r, :] (also written to sum_out)
hipError_t launch_rms_norm(const void* x, const void* addend, const void* scale,
                           void* sum_out, void* out, int64_t rows, int width,
                           float eps, int dtype, hipStream_t s);
// Steps of the local-attention block around its matrix products
// (rg_attention.hip).
hipError_t launch_rope(const void* x, const void* pos, int pos_kind,
                       const float* inv_freq, void* out, int64_t rows, int n,
                       int hd, const void* x2, void* out2, int n2, int dtype,
                       hipStream_t s);
hipError_t launch_attn_decode_probs(const void* scores, const void* q,
                                    const void* k_new,
                                    const int32_t* num_tokens, void* probs,
                                    int B, int heads, int hd, int window,
                                    float scale, int dtype, hipStream_t s);
hipError_t launch_attn_decode_finish(const void* from_ring, const void* probs,
                                     const void* k_new, const void* v_new,
                                     void* out, void* ring_k, void* ring_v,
                                     int32_t* num_tokens, int B, int heads,
                                     int hd, int window, int update, int dtype,
                                     hipStream_t s);
// Linear layers for at most 64 rows (rg_linear.hip).
int linear_rows_k_slices(int K, int N);
hipError_t launch_linear_pack(const void* w, void* packed, int N, int K,
                              int layout, int groups, int pair, hipStream_t s);
hipError_t launch_linear_rows(const LinearArgs& a, int gelu_pair,
                              hipStream_t s);
hipError_t launch_linear_rows_beside(const LinearArgs& a, hipStream_t s);
// Only the fp32 partial sums a.partial[slices][M][N] of x @ W^T, K split in
// `slices`; rg_elementwise.hip's norm kernel takes them from there.
bool block_step_f32_serves(const StepF32Args& a);
hipError_t launch_block_step_f32(const StepF32Args& a, hipStream_t s);
bool linear_rows_normed_serve(int M, int K, int N, int gelu_pair);
hipError_t launch_linear_rows_normed(const NormedLinearArgs& a, int gelu_pair,
                                     hipStream_t s);
hipError_t launch_linear_rows_partial(const LinearArgs& a, int slices,
                                      hipStream_t s);
hipError_t launch_add_rms_norm_runs(const void* x, const void* addend, const void* scale,
                                    void* sum_out, void* out, const int* runs, int count,
                                    int width, float eps, hipStream_t s);
hipError_t launch_rms_norm_partial(const float* sums, int slices,
                                   const void* bias, const void* addend,
                                   const void* scale, void* sum_out, void* out,
                                   int rows, int width, float eps,
                                   hipStream_t s);
// out[0] = shader cycles, out[1] = 10 ns ticks that `iters` rounds of a short
// dependent instruction chain took (rg_elementwise.hip)
hipError_t launch_clock_probe(uint64_t* out, int iters, hipStream_t s);
// rg_train.hip: the rest of a training step's backward pass.
// dx += dgx W_x^T + dga W_a^T per head (bf16, 256-wide heads)
hipError_t launch_gates_dgrad(const void* dgx, const void* dga, const void* w_x,
                              const void* w_a, void* dx, int64_t M, int W, int H,
                              hipStream_t s);
// rows per partial sum of the column sums below
constexpr int kColSumRows = 64;
// partial[ceil(M / kColSumRows)][W] of in [M, W] (W a multiple of 16 bytes)
hipError_t launch_col_sums(const void* in, float* partial, int64_t M, int W,
                           int dtype, hipStream_t s);
// launch_gelu_mul_backward and the column sums of d_g in one pass
hipError_t launch_gelu_mul_backward_sums(const void* dout, const void* a,
                                         const void* g, void* d_a, void* d_g,
                                         float* partial, int64_t M, int W,
                                         int dtype, hipStream_t s);
// out[n] = sum over rows of in[row * ld + n], rounded once; several at a time
struct SumTask {
  const float* in;
  int rows, n, ld;
  void* out;
};
constexpr int kMaxSumTasks = 8;
hipError_t launch_sum_rows(const SumTask* tasks, int count, int dtype,
                           hipStream_t s);
// rg_gates_split_f32.hip: both gate projections in float32 (256-wide heads; biases:
// both or neither); what they give back to x, added to dx; the gradients of their
// weights (workspace may be null where that needs no bytes).
bool gates_f32_serves(int64_t M, int W, int H);
hipError_t launch_gates_f32(const void* x, const void* w_x, const void* w_a,
                            const void* b_x, const void* b_a, void* gx, void* ga,
                            int64_t M, int W, int H, hipStream_t s);
hipError_t launch_gates_dgrad_f32(const void* dgx, const void* dga,
                                  const void* w_x, const void* w_a, void* dx,
                                  int64_t M, int W, int H, hipStream_t s);
bool gates_wgrad_f32_serves(int64_t M, int W, int H);
size_t gates_wgrad_f32_workspace_bytes(int64_t M, int W, int H);
hipError_t launch_gates_wgrad_f32(const void* x, const void* dgx,
                                  const void* dga, void* dwx, void* dwa,
                                  void* workspace, int64_t M, int W, int H,
                                  hipStream_t s);

// rg_gates_wgrad.hip: weight and bias gradients of both gate projections
bool gates_wgrad_serves(int64_t M, int W, int H);
size_t gates_wgrad_workspace_bytes(int64_t M, int W, int H);
hipError_t launch_gates_wgrad(const void* x, const void* dgx, const void* dga,
                              void* dwx, void* dwa, void* dbx, void* dba,
                              void* workspace, int64_t M, int W, int H,
                              hipStream_t s);
// bf16 [H,bw,bw] x 2 -> one buffer in MFMA operand order (head, group of 32
// channels, k-step, gate, lane, 8 values), zeros beyond bw.
int gate_k_steps(int bw);
size_t packed_gate_weights_bytes(int W, int H);
hipError_t launch_pack_gate_weights(const void* w_x, const void* w_a,
                                    void* packed, int W, int H, hipStream_t s);

}  // namespace rg
#endif  // RG_INTERNAL_H_
