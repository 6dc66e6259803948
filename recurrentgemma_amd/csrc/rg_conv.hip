// Stand-alone Conv1D kernels (any temporal width): the module-level drop-in
// for Conv1D.forward.  The fused prefill path does the width-4 conv inside the
// gate GEMM and the scan kernel instead and does not come through here.
#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

// One thread per output element; consecutive threads take consecutive
// channels, so every tap is a coalesced row read (taps hit L2 after the first).
template <typename T>
__global__ void __launch_bounds__(256)
conv1d_prefill_kernel(const T* __restrict__ x, const void* __restrict__ segpos,
                      int seg_kind, const T* __restrict__ w,
                      const T* __restrict__ bias, T* __restrict__ out,
                      int T_len, int W, int K, int64_t total) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; idx < total; idx += stride) {
    const int64_t m = idx / W;
    const int c = (int)(idx - m * W);
    store_scalar(out + idx,
                 conv_point<T>(x, segpos, seg_kind, w, bias, T_len, W, K, m, c));
  }
}

// The conv state the reference hands back after a prefill: the last K-1 input
// rows, each zeroed if a document starts in one of the (up to K-1) positions
// after it; rows before the start of the sequence are zero.
template <typename T>
__global__ void __launch_bounds__(256)
conv1d_cache_tail_kernel(const T* __restrict__ x,
                         const void* __restrict__ segpos, int seg_kind,
                         T* __restrict__ cache_out, int B, int T_len, int W,
                         int K) {
  const int64_t total = (int64_t)B * (K - 1) * W;
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; idx < total; idx += stride) {
    const int c = (int)(idx % W);
    const int64_t bk = idx / W;
    const int k = (int)(bk % (K - 1));
    const int64_t b = bk / (K - 1);
    const int t = T_len - (K - 1) + k;
    float v = 0.0f;
    if (t >= 0) {
      bool alive = true;
      for (int j = 1; j <= K - 1 && t + j <= T_len - 1; ++j)
        if (is_doc_start(segpos, seg_kind, b * T_len + t + j)) alive = false;
      if (alive) v = load_scalar(x + (b * T_len + t) * W + c);
    }
    store_scalar(cache_out + idx, v);
  }
}

// Backward pass of the prefill conv.  With keep_s[t] = "no document starts
// among tokens t-s+1 .. t" (what conv_point applies tap by tap):
//   out[t] = bias + sum_s w[K-1-s] x[t-s] keep_s[t]
//   dx[u]      = sum_s w[K-1-s] dout[u+s] keep_s[u+s]        (u + s < T)
//   dw[K-1-s] += x[t-s] keep_s[t] dout[t],   dbias += dout[t]
// A thread owns one channel and a run of `rows` consecutive flattened rows
// (b, t): it writes dx for them and leaves its sums of dw and dbias in
// `partial` [row chunks][K + 1][W] (float32), which the caller adds up.  The
// neighbouring rows it re-reads come from cache.  `rows` is 32 while that
// leaves at most 512 chunks and grows up to 256 beyond (conv1d_backward_rows):
// a plane of partial sums is (K + 1) W floats written and read again, 16 %
// of the pass's own traffic at 32 rows of bf16 and 2 % at 256.
constexpr int kConvBwdRows = 32;
constexpr int kConvBwdMaxRows = 256;
constexpr int kConvBwdChunks = 512;

template <typename T>
__global__ void __launch_bounds__(256)
conv1d_backward_kernel(const T* __restrict__ dout, const T* __restrict__ x,
                       const void* __restrict__ segpos, int seg_kind,
                       const T* __restrict__ w, T* __restrict__ dx,
                       float* __restrict__ partial, int T_len, int W, int K,
                       int64_t M, int rows) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= W) return;
  const int64_t m0 = (int64_t)blockIdx.x * rows;
  const int64_t m1 = m0 + rows < M ? m0 + rows : M;
  constexpr int kMaxK = 16;  // widths above are refused by the caller
  float wk[kMaxK], dw[kMaxK], db = 0.0f;
#pragma unroll
  for (int s = 0; s < kMaxK; ++s) {
    wk[s] = s < K ? load_scalar(w + (int64_t)(K - 1 - s) * W + c) : 0.0f;
    dw[s] = 0.0f;
  }
  for (int64_t m = m0; m < m1; ++m) {
    const int t = (int)(m % T_len);
    const float g = load_scalar(dout + m * W + c);
    db += g;
    float acc = 0.0f;
    bool back = true, ahead = true;
#pragma unroll
    for (int s = 0; s < kMaxK; ++s) {
      if (s < K) {
        // tap s of token t looks back at x[t-s]
        if (s > 0 && s <= t && is_doc_start(segpos, seg_kind, m - s + 1))
          back = false;
        if (s <= t && back)
          dw[s] = __builtin_fmaf(load_scalar(x + (m - s) * W + c), g, dw[s]);
        // token t is x[t'-s] of token t' = t + s
        if (s > 0 && t + s < T_len && is_doc_start(segpos, seg_kind, m + s))
          ahead = false;
        if (t + s < T_len && ahead)
          acc = __builtin_fmaf(wk[s], load_scalar(dout + (m + s) * W + c), acc);
      }
    }
    store_scalar(dx + m * W + c, acc);
  }
  float* out = partial + (int64_t)blockIdx.x * (K + 1) * W + c;
#pragma unroll
  for (int s = 0; s < kMaxK; ++s)
    if (s < K) out[(int64_t)(K - 1 - s) * W] = dw[s];
  out[(int64_t)K * W] = db;
}

// ---- temporal width 4, 16 bytes per lane: the usual case, streaming ---------
// A wave takes 32 consecutive flattened rows (b, t) of 64 x 16 bytes of
// channels; a lane walks its rows in time order with the three rows before the
// current one in registers (loaded once as a halo), so every row of x is read
// once (plus 3 in 32 for the halo) and every output row written once, as
// 16-byte accesses.  A document start -- or the first token of a sequence row --
// zeroes the history registers: later tokens then see zeros exactly where the
// definition drops a tap.  Rows are requested eight at a time before the first
// is used.
constexpr int kConvRun = 32;    // rows per wave of the forward kernels
constexpr int kConvBatch = 8;   // rows requested together
constexpr int kConvFlagRows = 48;  // rows between two looks at 64 rows' flags

template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
  static constexpr int N = 4;
  __device__ static void unpack(u32x4 r, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(r[i]);
  }
  __device__ static u32x4 pack(const float (&v)[4]) {
    return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]),
                 __float_as_uint(v[2]), __float_as_uint(v[3])};
  }
};
template <>
struct Vec16<uint16_t> {
  static constexpr int N = 8;
  __device__ static void unpack(u32x4 r, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(r[i] << 16);
      v[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
  __device__ static u32x4 pack(const float (&v)[8]) {
    return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                 pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
  }
};
// four channels of a lane, whatever they are stored as
template <typename T>
struct Vec4ch : Vec16<float> {
  typedef u32x4 Raw;
};
template <>
struct Vec4ch<uint16_t> {
  static constexpr int N = 4;
  typedef u32x2 Raw;
  __device__ static void unpack(u32x2 r, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      v[2 * i] = __uint_as_float(r[i] << 16);
      v[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
  __device__ static u32x2 pack(const float (&v)[4]) {
    return u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
};

// Which of the rows around a run (fewer than `span` of them, from `base` on)
// is the first token of a sequence row: at most one when the sequences are at
// least `span` tokens long, found once per wave instead of a 64-bit remainder
// per row.
struct SeqStarts {
  int64_t first;  // first row >= base that begins a sequence row
  int T_len;
  bool one;       // the sequences are long enough for `first` to be the only one
  __device__ SeqStarts(int64_t base, int T, int span) : T_len(T), one(T >= span) {
    const int64_t r = base % T;
    first = r == 0 ? base : base + (T - r);
  }
  __device__ bool at(int64_t m) const {
    return one ? m == first : m % T_len == 0;
  }
};

// row m starts a history: first token of a sequence row, or of a document
__device__ __forceinline__ bool conv_row_starts(const void* segpos, int seg_kind,
                                                const SeqStarts& seq, int64_t m) {
  return seq.at(m) || is_doc_start(segpos, seg_kind, m);
}

// The same for the 64 rows from `base` on, a bit each, rows behind the last one (M - 1)
// among the starts: a lane a row and one load, where a test of a flag row by row is a
// branch and a wait for everything the wave has asked for.  Every lane of the wave takes
// part.
__device__ __forceinline__ uint64_t start_bits(const void* segpos, int seg_kind,
                                               int64_t base, int T_len, int64_t M) {
  const int64_t m = base + ((int)threadIdx.x & 63);
  bool starts = m >= M;
  if (m >= 0 && m < M) starts = m % T_len == 0 || is_doc_start(segpos, seg_kind, m);
  return __ballot(starts);
}

// RUN rows per wave: the longer, the fewer halo rows are read twice (3 per
// run) and the fewer workgroups are dispatched.  The blocks behind the runs, one
// for every sequence, write its conv state (conv1d_cache_tail_kernel's).
template <typename T, int RUN>
__global__ void __launch_bounds__(1024)
conv1d_prefill_k4_kernel(const T* __restrict__ x, const void* __restrict__ segpos,
                         int seg_kind, const T* __restrict__ w,
                         const T* __restrict__ bias, T* __restrict__ out,
                         T* __restrict__ cache_out, int T_len, int W, int64_t M) {
  using V = Vec16<T>;
  constexpr int N = V::N;
  // the waves of a workgroup lie side by side along a row (up to 16 of them:
  // 16 KB of a row), so that what they request together is contiguous
  const int own_c = ((int)blockIdx.y * (int)blockDim.x + (int)threadIdx.x) * N;
  // (W % N == 0: a lane is inside or outside; those outside do the last one's work once
  // more, with its values, beside lanes inside: every lane has a row's flag to load)
  if (own_c - ((int)threadIdx.x & 63) * N >= W) return;
  const int c = own_c < W ? own_c : W - N;
  const int64_t m0 = (int64_t)blockIdx.x * RUN;
  if (m0 >= M) {
    const int64_t b = (int64_t)blockIdx.x - (M + RUN - 1) / RUN;
    bool cut = false;  // a document starts behind the row
#pragma unroll
    for (int k = 2; k >= 0; --k) {
      const int t = T_len - 3 + k;
      u32x4 v = {0, 0, 0, 0};
      if (t >= 0 && !cut)
        v = *reinterpret_cast<const u32x4*>(x + (b * T_len + t) * W + c);
      *reinterpret_cast<u32x4*>(cache_out + (b * 3 + k) * W + c) = v;
      if (t >= 0 && is_doc_start(segpos, seg_kind, b * T_len + t)) cut = true;
    }
    return;
  }
  const int64_t m1 = m0 + RUN < M ? m0 + RUN : M;
  auto row = [&](const T* base, int64_t m) {
    return *reinterpret_cast<const u32x4*>(base + m * W + c);
  };
  if constexpr (sizeof(T) == 2) {
    // bf16: the kernels' one width-4 arithmetic (conv4_dot of rg_common.h) on
    // rows that stay packed: per channel the time pairs (x[t-1], x[t]), two
    // dot products per output.  No branch lies between the loads: the starts are bits, and
    // the row eight on takes the place of the one that is used up.  us, with a look at the
    // flags row by row before: B1 T64 W2560 5.5 -> 4.0, B1 T512 6.7 -> 4.6, B4 T2048 22.9
    // -> 21.3, B16 T4096 138 -> 132.  (Float32 so: 5.3 -> 4.1, 6.3 -> 5.1 and 39.1 -> 38.3,
    // but B3 T2048 29.0 -> 31.2 and 2 to 3 % at B3 T1001, B2 T2048: left as it was.)
    u32x4 before[3], raw[kConvBatch];
#pragma unroll
    for (int k = 0; k < 3; ++k) before[k] = row(x, m0 ? m0 - 3 + k : 0);
#pragma unroll
    for (int u = 0; u < kConvBatch; ++u) raw[u] = row(x, m0 + u < m1 ? m0 + u : m1 - 1);
    uint64_t bits = start_bits(segpos, seg_kind, m0 - 3, T_len, M);  // bit 0: the next row
    float bb[N];
    V::unpack(*reinterpret_cast<const u32x4*>(bias + c), bb);
    uint32_t w10[N], w32[N];
    {
      const u32x4 t0 = row(w, 0), t1 = row(w, 1), t2 = row(w, 2), t3 = row(w, 3);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        pair_up(t0[q], t1[q], w10[2 * q], w10[2 * q + 1]);
        pair_up(t2[q], t3[q], w32[2 * q], w32[2 * q + 1]);
      }
    }
    // history: the row before (packed) and the pairs that ended one and two
    // rows back; zero where a start cuts
    u32x4 r1 = {0, 0, 0, 0};
    uint32_t pn1[N], pn2[N];
#pragma unroll
    for (int e = 0; e < N; ++e) pn1[e] = pn2[e] = 0u;
    auto cut = [&]() {
      r1 = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < N; ++e) pn1[e] = pn2[e] = 0u;
    };
    auto push = [&](const u32x4& cur, uint32_t (&pn0)[N]) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        pair_up(r1[q], cur[q], pn0[2 * q], pn0[2 * q + 1]);
    };
    auto shift = [&](const u32x4& cur, const uint32_t (&pn0)[N]) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        pn2[e] = pn1[e];
        pn1[e] = pn0[e];
      }
      r1 = cur;
    };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (m0) {
        if (bits & 1) cut();
        uint32_t pn0[N];
        push(before[k], pn0);
        shift(before[k], pn0);
      }
      bits >>= 1;
    }
    auto one_row = [&](int64_t m, const u32x4& cur) __attribute__((always_inline)) {
      if (bits & 1) cut();
      bits >>= 1;
      uint32_t pn0[N];
      push(cur, pn0);
      float o[N];
#pragma unroll
      for (int q = 0; q < N; q += 4) {
        const uint32_t po[4] = {pn2[q], pn2[q + 1], pn2[q + 2], pn2[q + 3]};
        const uint32_t pw[4] = {pn0[q], pn0[q + 1], pn0[q + 2], pn0[q + 3]};
        const uint32_t wa[4] = {w10[q], w10[q + 1], w10[q + 2], w10[q + 3]};
        const uint32_t wb[4] = {w32[q], w32[q + 1], w32[q + 2], w32[q + 3]};
        const float bq[4] = {bb[q], bb[q + 1], bb[q + 2], bb[q + 3]};
        float oq[4];
        conv4_dot_x4(po, pw, wa, wb, bq, oq);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[q + e] = oq[e];
      }
      shift(cur, pn0);
      *reinterpret_cast<u32x4*>(out + m * W + c) = V::pack(o);
    };
    auto look = [&](int64_t mb) __attribute__((always_inline)) {
      if (RUN > kConvFlagRows && mb > m0 && (mb - m0) % kConvFlagRows == 0)
        bits = start_bits(segpos, seg_kind, mb, T_len, M);
    };
    int64_t mb = m0;
    for (; mb + kConvBatch <= m1; mb += kConvBatch) {
      look(mb);
#pragma unroll
      for (int u = 0; u < kConvBatch; ++u) {
        one_row(mb + u, raw[u]);
        const int64_t ahead = mb + u + kConvBatch;
        if (RUN > kConvBatch) raw[u] = row(x, ahead < m1 ? ahead : m1 - 1);
      }
    }
    if (mb < m1) {
      look(mb);
#pragma unroll
      for (int u = 0; u < kConvBatch; ++u)
        if (mb + u < m1) one_row(mb + u, raw[u]);
    }
    return;
  }
  const SeqStarts seq(m0 >= 3 ? m0 - 3 : 0, T_len, RUN + 3);
  float w0[N], w1[N], w2[N], w3[N], bb[N];
  V::unpack(row(w, 0), w0);
  V::unpack(row(w, 1), w1);
  V::unpack(row(w, 2), w2);
  V::unpack(row(w, 3), w3);
  V::unpack(*reinterpret_cast<const u32x4*>(bias + c), bb);
  // history: h1 = x[m-1], h2 = x[m-2], h3 = x[m-3], zero where a start cuts
  float h1[N], h2[N], h3[N];
#pragma unroll
  for (int e = 0; e < N; ++e) h1[e] = h2[e] = h3[e] = 0.0f;
  for (int64_t j = m0 - 3; j < m0; ++j) {
    if (j < 0) continue;
    if (conv_row_starts(segpos, seg_kind, seq, j)) {
#pragma unroll
      for (int e = 0; e < N; ++e) h1[e] = h2[e] = 0.0f;
    }
#pragma unroll
    for (int e = 0; e < N; ++e) {
      h3[e] = h2[e];
      h2[e] = h1[e];
    }
    V::unpack(row(x, j), h1);
  }
  for (int64_t mb = m0; mb < m1; mb += kConvBatch) {
    u32x4 raw[kConvBatch];
    bool st[kConvBatch];
#pragma unroll
    for (int u = 0; u < kConvBatch; ++u) {
      const int64_t m = mb + u < m1 ? mb + u : m1 - 1;
      raw[u] = row(x, m);
      st[u] = conv_row_starts(segpos, seg_kind, seq, m);
    }
#pragma unroll
    for (int u = 0; u < kConvBatch; ++u) {
      if (mb + u < m1) {
        if (st[u]) {
#pragma unroll
          for (int e = 0; e < N; ++e) h1[e] = h2[e] = h3[e] = 0.0f;
        }
        float cur[N], o[N];
        V::unpack(raw[u], cur);
#pragma unroll
        for (int e = 0; e < N; ++e) {
          o[e] = conv4(cur[e], h1[e], h2[e], h3[e], w0[e], w1[e], w2[e], w3[e],
                       bb[e]);
          h3[e] = h2[e];
          h2[e] = h1[e];
          h1[e] = cur[e];
        }
        *reinterpret_cast<u32x4*>(out + (mb + u) * W + c) = V::pack(o);
      }
    }
  }
}

// The backward pass in the same shape: the window of x slides as above (for
// dw), a window of dout[m .. m+3] slides ahead of it (for dx), with the starts
// of rows m+1 .. m+3 deciding which of them a tap may use.  Sums for dw and
// dbias go to the chunk's plane of `partial` like the general kernel's.
//
// A chunk's rows are shared by the WAVES waves of a workgroup, whose sums meet in LDS.
// What bounds it: memory from some 30 us on, the way of the first rows before that.  A
// lane has four channels, so that three waves a SIMD have registers (137 of them; with
// eight channels of bf16 247, two waves and 5 waves for 4 SIMDs at B4 T2048 W2560), and a
// row's loads are asked for as the row eight (float32: four) in front of it is used up:
// no branch lies between them, the flags are bits.  bf16 B4 T2048 W2560 with operands in
// memory: 45 us with a look at the flags row by row, eight channels a lane and a batch of
// rows waited for at a time; 38 with the bits and loads one by one; 34 with four channels
// (139 MB: 4.1 TB/s).  Float32 60 either way, 8.5 -> 7.0 at B1 T300.
template <typename T, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 3)
conv1d_backward_k4_kernel(const T* __restrict__ dout, const T* __restrict__ x,
                          const void* __restrict__ segpos, int seg_kind,
                          const T* __restrict__ w, T* __restrict__ dx,
                          float* __restrict__ partial,
                          float* __restrict__ dx_sums, int T_len, int W,
                          int64_t M, int rows) {
  using V = Vec4ch<T>;
  using Raw = typename V::Raw;
  constexpr int N = V::N;
  constexpr int kBatch = sizeof(T) == 4 ? 4 : 8;  // rows on their way
  __shared__ float others[WAVES > 1 ? WAVES - 1 : 1][WAVES > 1 ? 6 * N : 1][64];
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // (lanes behind a row's end do the last one's work once more, with its values: every
  // lane has a row's flag to load)
  const int own_c = ((int)blockIdx.y * 64 + lane) * N;
  const int c = own_c < W ? own_c : W - N;
  const int share = rows / WAVES;
  const int64_t m0 = (int64_t)blockIdx.x * rows + wave * share;
  const int64_t m1 = m0 + share < M ? m0 + share : M;
  float d0[N], d1[N], d2[N], d3[N], db[N], dxs[N];
#pragma unroll
  for (int e = 0; e < N; ++e)
    d0[e] = d1[e] = d2[e] = d3[e] = db[e] = dxs[e] = 0.0f;
  if (WAVES == 1 || m0 < M) {
    auto row = [&](const T* base, int64_t m) {
      return *reinterpret_cast<const Raw*>(base + m * W + c);
    };
    // (rows outside: any row inside, not used)
    auto row_in = [&](const T* base, int64_t m) {
      return row(base, m < 0 ? 0 : m < M ? m : M - 1);
    };
    Raw taps[4], before[3], after[3], xr[kBatch], gr[kBatch];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      before[k] = row_in(x, m0 - 1 - k);
      after[k] = row_in(dout, m0 + k);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) taps[k] = row(w, k);
    // bit 0: row m0 (or the row that begins the present kConvFlagRows)
    uint64_t bits = start_bits(segpos, seg_kind, m0 - 3, T_len, M);
    const bool cut1 = (bits >> 2) & 1, cut2 = cut1 || ((bits >> 1) & 1);
    bits >>= 3;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      xr[u] = row_in(x, m0 + u);
      gr[u] = row_in(dout, m0 + u + 3);
    }
    float w0[N], w1[N], w2[N], w3[N];
    V::unpack(taps[0], w0);
    V::unpack(taps[1], w1);
    V::unpack(taps[2], w2);
    V::unpack(taps[3], w3);
    // the rows before, as far as no start cuts them off; g0 = dout[m], g1 .. g3 the
    // rows after it
    float h1[N], h2[N], h3[N], g0[N], g1[N], g2[N], g3[N];
    auto take = [](bool used, const Raw& r, float (&v)[N]) {
      V::unpack(used ? r : Raw(0u), v);
    };
    // (m0 is 0 or 8 at least)
    take(m0 > 0, before[0], h1);
    take(m0 > 0 && !cut1, before[1], h2);
    take(m0 > 0 && !cut2, before[2], h3);
    V::unpack(after[0], g0);
    V::unpack(after[1], g1);
    V::unpack(after[2], g2);
    auto one_row = [&](int64_t m, const Raw& xm, const Raw& gm)
        __attribute__((always_inline)) {
      float cur[N], o[N];
      V::unpack(xm, cur);
      V::unpack(gm, g3);
      if (bits & 1) {
#pragma unroll
        for (int e = 0; e < N; ++e) h1[e] = h2[e] = h3[e] = 0.0f;
      }
      // a tap reaches the rows of dout in front of the next start
      const bool ok1 = !(bits & 2), ok2 = !(bits & 6), ok3 = !(bits & 14);
      bits >>= 1;
#pragma unroll
      for (int e = 0; e < N; ++e) {
        float acc = w3[e] * g0[e];
        acc = __builtin_fmaf(w2[e], ok1 ? g1[e] : 0.0f, acc);
        acc = __builtin_fmaf(w1[e], ok2 ? g2[e] : 0.0f, acc);
        acc = __builtin_fmaf(w0[e], ok3 ? g3[e] : 0.0f, acc);
        o[e] = acc;
        d3[e] = __builtin_fmaf(cur[e], g0[e], d3[e]);  // w[3] meets x[t]
        d2[e] = __builtin_fmaf(h1[e], g0[e], d2[e]);
        d1[e] = __builtin_fmaf(h2[e], g0[e], d1[e]);
        d0[e] = __builtin_fmaf(h3[e], g0[e], d0[e]);
        db[e] += g0[e];
        h3[e] = h2[e];
        h2[e] = h1[e];
        h1[e] = cur[e];
        g0[e] = g1[e];
        g1[e] = g2[e];
        g2[e] = g3[e];
      }
      const Raw packed = V::pack(o);
      *reinterpret_cast<Raw*>(dx + m * W + c) = packed;
      // (of what is stored: the bias gradient of the layer in front)
      V::unpack(packed, o);
#pragma unroll
      for (int e = 0; e < N; ++e) dxs[e] += o[e];
    };
    int64_t mb = m0;
    // whole batches, without a branch around a load: the row eight on takes the place of
    // the one that has been used (behind the last one the last once more)
    for (; mb + kBatch <= m1; mb += kBatch) {
      if (mb > m0 && (mb - m0) % kConvFlagRows == 0)
        bits = start_bits(segpos, seg_kind, mb, T_len, M);
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int64_t m = mb + u, ahead = m + kBatch < m1 ? m + kBatch : m1 - 1;
        one_row(m, xr[u], gr[u]);
        xr[u] = row(x, ahead);
        gr[u] = row(dout, ahead + 3 < M ? ahead + 3 : M - 1);
      }
    }
    if (mb < m1) {
      if (mb > m0 && (mb - m0) % kConvFlagRows == 0)
        bits = start_bits(segpos, seg_kind, mb, T_len, M);
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (mb + u < m1) one_row(mb + u, xr[u], gr[u]);
    }
  }
  if constexpr (WAVES > 1) {
    auto meet = [&](int i, float (&v)[N]) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        if (wave > 0) {
          others[wave - 1][i * N + e][lane] = v[e];
        } else {
#pragma unroll
          for (int k = 0; k < WAVES - 1; ++k) v[e] += others[k][i * N + e][lane];
        }
      }
    };
    auto meet_all = [&]() {
      meet(0, d0);
      meet(1, d1);
      meet(2, d2);
      meet(3, d3);
      meet(4, db);
      meet(5, dxs);
    };
    if (wave > 0) meet_all();
    __syncthreads();
    if (wave > 0) return;
    meet_all();
  }
  if (own_c >= W) return;
  if (dx_sums != nullptr) {
#pragma unroll
    for (int e = 0; e < N; ++e) dx_sums[(int64_t)blockIdx.x * W + c + e] = dxs[e];
  }
  float* outp = partial + (int64_t)blockIdx.x * 5 * W + c;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    outp[e] = d0[e];
    outp[(int64_t)W + e] = d1[e];
    outp[2 * (int64_t)W + e] = d2[e];
    outp[3 * (int64_t)W + e] = d3[e];
    outp[4 * (int64_t)W + e] = db[e];
  }
}

// Decode step: one thread per (batch row, channel).  All state rows are read
// into registers before anything is written, so cache_out may alias cache_in.
template <typename T>
__global__ void __launch_bounds__(256)
conv1d_step_kernel(const T* __restrict__ x, const T* cache_in,
                   const T* __restrict__ w, const T* __restrict__ bias,
                   T* __restrict__ out, T* cache_out, int B, int W, int K) {
  const int64_t total = (int64_t)B * W;
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; idx < total; idx += stride) {
    const int c = (int)(idx % W);
    const int64_t b = idx / W;
    float st[16];  // K - 1 <= 15 state rows, oldest first
#pragma unroll
    for (int k = 0; k < 15; ++k)
      st[k] = (k < K - 1) ? load_scalar(cache_in + (b * (K - 1) + k) * W + c)
                          : 0.0f;
    const float xv = load_scalar(x + idx);
    float acc;
    if (sizeof(T) == 2 && K == 4) {
      // the bf16 kernels' width-4 arithmetic (conv4_dot of rg_common.h)
      acc = conv4_bf16(xv, st[2], st[1], st[0], load_scalar(w + c),
                       load_scalar(w + (int64_t)W + c),
                       load_scalar(w + 2 * (int64_t)W + c),
                       load_scalar(w + 3 * (int64_t)W + c),
                       load_scalar(bias + c));
    } else {
      acc = load_scalar(bias + c);
      acc = __builtin_fmaf(xv, load_scalar(w + (int64_t)(K - 1) * W + c), acc);
#pragma unroll
      for (int k = 14; k >= 0; --k)  // newest state row first
        if (k < K - 1)
          acc = __builtin_fmaf(st[k], load_scalar(w + (int64_t)k * W + c), acc);
    }
    store_scalar(out + idx, acc);
    if (cache_out) {
#pragma unroll
      for (int k = 0; k < 15; ++k)
        if (k < K - 2) store_scalar(cache_out + (b * (K - 1) + k) * W + c,
                                    st[k + 1]);
      store_scalar(cache_out + (b * (K - 1) + (K - 2)) * W + c, xv);
    }
  }
}

inline int grid_for(int64_t total, int block) {
  int64_t g = (total + block - 1) / block;
  const int64_t cap = 256 * 64;  // grid-stride loop beyond this
  return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

// whether the 16-byte kernels serve this shape
template <typename T>
bool conv_k4_fits(int K, int W, int64_t M) {
  constexpr int N = 16 / (int)sizeof(T);
  return K == 4 && W % N == 0 && (M + kConvRun - 1) / kConvRun <= 0x7fffffff &&
         (W / N + 63) / 64 <= 65535;
}

template <typename T>
hipError_t conv_prefill_t(const ConvArgs& a, hipStream_t s) {
  const int64_t total = (int64_t)a.B * a.T * a.W;
  const int64_t M = (int64_t)a.B * a.T;
  if (conv_k4_fits<T>(a.K, a.W, M)) {
    constexpr int N = 16 / (int)sizeof(T);
    const unsigned slabs = (unsigned)((a.W / N + 63) / 64);
    const unsigned waves = slabs < 16 ? slabs : 16;  // per workgroup
    const unsigned across = (slabs + waves - 1) / waves;
    const int tails = a.cache_out ? a.B : 0;
    auto launch = [&](auto RUN) {
      constexpr int run = decltype(RUN)::value;
      const dim3 grid((unsigned)((M + run - 1) / run + tails), across);
      conv1d_prefill_k4_kernel<T, run><<<grid, waves * 64, 0, s>>>(
          (const T*)a.x, a.segpos, a.seg_kind, (const T*)a.w, (const T*)a.bias,
          (T*)a.out, (T*)a.cache_out, a.T, a.W, M);
    };
    // long runs where that still leaves eight waves for every SIMD, short ones
    // where runs of 32 leave fewer than two: a run's rows come eight at a time,
    // one memory round trip after the other (B1 T512 W2560 float32: 16 us, 8 rows
    // 6)
    constexpr int kLongRun = 128, kShortRun = 8;
    if ((M / kLongRun) * slabs >= 8192)
      launch(std::integral_constant<int, kLongRun>{});
    else if ((M / kConvRun) * slabs >= 2048)
      launch(std::integral_constant<int, kConvRun>{});
    else
      launch(std::integral_constant<int, kShortRun>{});
    return hipGetLastError();
  }
  conv1d_prefill_kernel<T><<<grid_for(total, 256), 256, 0, s>>>(
      (const T*)a.x, a.segpos, a.seg_kind, (const T*)a.w, (const T*)a.bias,
      (T*)a.out, a.T, a.W, a.K, total);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !a.cache_out) return e;
  const int64_t ctotal = (int64_t)a.B * (a.K - 1) * a.W;
  conv1d_cache_tail_kernel<T><<<grid_for(ctotal, 256), 256, 0, s>>>(
      (const T*)a.x, a.segpos, a.seg_kind, (T*)a.cache_out, a.B, a.T, a.W,
      a.K);
  return hipGetLastError();
}

template <typename T>
hipError_t conv_step_t(const ConvStepArgs& a, hipStream_t s) {
  const int64_t total = (int64_t)a.B * a.W;
  conv1d_step_kernel<T><<<grid_for(total, 256), 256, 0, s>>>(
      (const T*)a.x, (const T*)a.cache_in, (const T*)a.w, (const T*)a.bias,
      (T*)a.out, (T*)a.cache_out, a.B, a.W, a.K);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_conv1d_prefill(const ConvArgs& a, int dtype, hipStream_t s) {
  return dtype == 0 ? conv_prefill_t<float>(a, s)
                    : conv_prefill_t<uint16_t>(a, s);
}

hipError_t launch_conv1d_step(const ConvStepArgs& a, int dtype,
                              hipStream_t s) {
  return dtype == 0 ? conv_step_t<float>(a, s) : conv_step_t<uint16_t>(a, s);
}

// Rows per chunk of the backward pass (see kConvBwdRows above).
static int conv1d_backward_rows(int64_t M) {
  int rows = kConvBwdRows;
  while (rows < kConvBwdMaxRows && (M + rows - 1) / rows > kConvBwdChunks)
    rows *= 2;
  return rows;
}

int conv1d_backward_chunks(int B, int T) {
  const int64_t M = (int64_t)B * T;
  const int rows = conv1d_backward_rows(M);
  return (int)((M + rows - 1) / rows);
}

bool conv1d_backward_sums_dx(int B, int T, int W, int K, int dtype) {
  const int64_t M = (int64_t)B * T;
  return dtype == 0 ? conv_k4_fits<float>(K, W, M) : conv_k4_fits<uint16_t>(K, W, M);
}

hipError_t launch_conv1d_backward(const ConvBwdArgs& a, int dtype,
                                  hipStream_t s) {
  const int64_t M = (int64_t)a.B * a.T;
  const int64_t chunks = conv1d_backward_chunks(a.B, a.T);
  const int rows = conv1d_backward_rows(M);
  const int64_t cblocks = ((int64_t)a.W + 255) / 256;
  if (chunks <= 0 || chunks > 0x7fffffff || cblocks > 65535 || a.K < 2 ||
      a.K > 16)
    return hipErrorInvalidValue;
  if (dtype == 0 ? conv_k4_fits<float>(a.K, a.W, M)
                 : conv_k4_fits<uint16_t>(a.K, a.W, M)) {
    // waves of a chunk: as many as there is room for on the CUs (us, one / two / four:
    // bf16 B1 T300 W2560 11.2 / 8.7 / 7.1, B1 T1000 13.5 / 10.4 / 9.2, B2 T1000 W4096
    // 17.3 / 16.6 / 18.5, B4 T2048 W2560 34.1 / 36.0 / 38.7, B8 T2048 W4096 103 / 111 /
    // 119; float32 12.1 / 8.8 / 7.0, 16.6 / 12.5 / 12.0, 27.3 / 25.4 / 29.8, 60.6 / 60.5 /
    // 61.0, 189 / 193 / 198)
    auto run = [&](auto* tag, auto waves) {
      typedef std::remove_pointer_t<decltype(tag)> T;
      constexpr int w = decltype(waves)::value;
      conv1d_backward_k4_kernel<T, w>
          <<<dim3((unsigned)chunks, (unsigned)((a.W / Vec4ch<T>::N + 63) / 64)), 64 * w,
             0, s>>>((const T*)a.dout, (const T*)a.x, a.segpos, a.seg_kind,
                     (const T*)a.w, (T*)a.dx, a.partial, a.dx_sums, a.T, a.W, M, rows);
    };
    auto pick = [&](auto* tag) {
      typedef std::remove_pointer_t<decltype(tag)> T;
      const int64_t blocks = chunks * ((a.W / Vec4ch<T>::N + 63) / 64);
      if (blocks <= 512) run(tag, std::integral_constant<int, 4>{});
      else if (blocks <= 1024) run(tag, std::integral_constant<int, 2>{});
      else run(tag, std::integral_constant<int, 1>{});
    };
    if (dtype == 0) pick((float*)nullptr);
    else pick((uint16_t*)nullptr);
    return hipGetLastError();
  }
  if (a.dx_sums != nullptr) return hipErrorInvalidValue;
  const dim3 grid((unsigned)chunks, (unsigned)cblocks);
  if (dtype == 0)
    conv1d_backward_kernel<float><<<grid, 256, 0, s>>>(
        (const float*)a.dout, (const float*)a.x, a.segpos, a.seg_kind,
        (const float*)a.w, (float*)a.dx, a.partial, a.T, a.W, a.K, M, rows);
  else
    conv1d_backward_kernel<uint16_t><<<grid, 256, 0, s>>>(
        (const uint16_t*)a.dout, (const uint16_t*)a.x, a.segpos, a.seg_kind,
        (const uint16_t*)a.w, (uint16_t*)a.dx, a.partial, a.T, a.W, a.K, M,
        rows);
  return hipGetLastError();
}

}  // namespace rg
