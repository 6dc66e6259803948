// The linear recurrence and the RG-LRU's gating around it, forward and
// backward, reading every element once: rnn_scan and RGLRU.forward of a
// training step (recurrentgemma/torch/layers.py:140-191, 335-360) and what
// autograd makes of them.
//
//   forward   h_t = a'_t h_{t-1} + x_t                      y_t = h_t
//   backward  g_t = dy_t + u_{t+1},  u_t = a'_t g_t         (from the end, the
//             dx_t = g_t,  da_t = g_t h_{t-1},  dh0 = u_0    incoming u is dh_last)
// with a' = a, zeroed at document starts.  Both are first-order recurrences
// on pairs (coefficient, input): (a', x) forwards, (a', a' dy) backwards.
//
// A lane owns 16 bytes of adjacent channels and KL consecutive tokens, a wave
// eight lanes of channels (128 bytes of a row) by eight groups of tokens, a
// workgroup of eight waves 64 groups: one step of 64 KL tokens.  Per step
//   1  every lane reduces its tokens, which stay in registers, to (P, H) per
//      channel;
//   2  the 64 pairs of a channel meet in LDS and are scanned by 512 / channels
//      threads, 64 channels / 8 pairs each, their totals by lane shifts (the
//      scan operator of recurrentgemma/jax/scan.py:161-187); the state that
//      comes into every group goes back through LDS;
//   3  every lane replays its tokens from that state and stores.
// Rows are asked for as early as the registers allow (see below), so that the
// memory pipe works while a step computes.
//
// A workgroup walks one slab of channels of one row, or (DEAL) the steps of all slabs
// are dealt out: few rows leave most CUs without a slab, and slabs beyond a multiple
// of the CUs take a round of their own.  One workgroup per CU takes steps from a
// counter, the first step of all slabs, then the second, ..; the state behind a step
// is one word per channel, value and number of the step, that goes through memory
// (agent-scope stores and loads of the whole word: no fence) to whoever has the next
// one, between that step's 2 and 3.  Two words per row and channel: the state of step
// s - 2 has been read when the one of s - 1 arrives.  Every wait ends: a workgroup
// works on its tickets in order, a step waits for one with a smaller ticket, and only
// a workgroup that runs takes tickets.  Sums over tokens leave a row per step.
// us, B1 T8192 W2560 bf16, slabs / dealt: plain forward 82 / 38, backward 130 / 49,
// gated 152 / 63 and 389 / 112; a step costs as much as before, the rest is the first
// launch (states and counter cleared), the first tickets and loads: 14 us.
// The kernels this replaces where it runs (rg_scan.hip, rg_scan_bwd.hip) keep
// one or two channels per lane: 80 .. 160 workgroups with 2- and 4-byte
// accesses at B4 W2560, and the backward ones read their inputs twice and
// evaluated the gates twice.
#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kLanes = 8;             // lanes side by side along the channels
constexpr int kGroups = kThreads / kLanes;  // token groups of a step

constexpr int kFwdPlain = kTilesFwdPlain, kBwdPlain = kTilesBwdPlain,
              kFwdGated = kTilesFwdGated, kBwdGated = kTilesBwdGated;
// cond ? a : b with both sides computed (the compiler would put the expensive
// one behind a branch per token, and split the replay into pieces that no load
// crosses).
__device__ __forceinline__ float choose(bool cond, float a, float b) {
  asm("" : "+v"(b));
  return cond ? a : b;
}

// 1 - a^2 for a = 2^q, q <= 0, in float32: near a = 1, where the difference of the
// rounded square would keep few of its digits, -q p(q) with p the polynomial of degree
// five through (2^2q - 1) / q at the Chebyshev nodes of -0.375 .. 0 (off by 2e-9 of it,
// as eight terms of the exponential's own series are by 2e-8).  With it the float32
// forms can use the hardware's exp2, reciprocal and square root (sigmoids: sigmoid_f32).
// Errors against 64 bits, projections included, before (expf, sqrtf and divisions) and
// now: gates around 0 y 1.0e-7 .. 1.6e-7 -> 7.2e-8 .. 1.2e-7, gradients 1.5e-7 ..
// 3.3e-7 -> 1.0e-7 .. 2.1e-7; input gates at -12 .. -8 y 4.0e-7 -> 3.4e-7; recurrence
// gates there y 4e-5 -> 6e-7.  Of this kernel alone (exact pre-activations): y and the
// gradients of x and the input gate as before, a_param's and the recurrence gate's bias
// up to 1.1 times for softplus(a_param) up to 1 (1.7e-7 -> 1.9e-7) and 1.5 times at 5,
// where a is e^-20.
__device__ __forceinline__ float one_minus_square(float q, float a) {
  constexpr float kNear[6] = {0.69314718246f * 0x1p1f,   0.24022640288f * 0x1p2f,
                              0.055502466857f * 0x1p3f,  0.0096086980775f * 0x1p4f,
                              0.0013086448889f * 0x1p5f, 0.00012355708168f * 0x1p6f};
  float s = kNear[5];
#pragma unroll
  for (int k = 4; k >= 0; --k) s = __builtin_fmaf(s, q, kNear[k]);
  return q > -0.375f ? -q * s : __builtin_fmaf(-a, a, 1.0f);
}

constexpr int streams_of(int mode) {
  return mode == kFwdPlain ? 2 : mode == kBwdGated ? 5 : 3;
}

template <typename T>
struct Vec;  // 16 bytes of channels
template <>
struct Vec<uint16_t> {
  static constexpr int n = 8;
  __device__ static void unpack(u32x4 r, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(r[i] << 16);
      v[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
  // rounded to the stored type (and v replaced by the rounded values)
  __device__ static u32x4 pack(float (&v)[8]) {
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    unpack(r, v);
    return r;
  }
};
template <>
struct Vec<float> {
  static constexpr int n = 4;
  __device__ static void unpack(u32x4 r, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(r[i]);
  }
  __device__ static u32x4 pack(float (&v)[4]) {
    return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]),
                 __float_as_uint(v[2]), __float_as_uint(v[3])};
  }
};

template <typename T>
struct TileLds {
  static constexpr int channels = kLanes * Vec<T>::n;
  // (two floats of padding: the scanning threads of a wave, whose first groups
  // lie channels / 8 rows apart, then start on different banks)
  float pair[kGroups][2 * channels + 2];  // P, H per channel
  float in[kGroups][channels + 4];        // state before the group
  // (dealt out: of this step's slab and the next one's)
  float sp[2][channels];                  // softplus of a_param
  float slope[2][channels];               // and its derivative
  float bias[2][2][channels];             // float32: of the gate projections
  int ticket[4];                          // dealt out: the last four
};

// What the dealt form has beside: states between steps, [B][2][W] words of value and
// number of the step; the tickets taken; total = steps x chains, chains = B x slabs.
struct DealArgs {
  uint64_t* words;
  float* soft;  // [2][W]: softplus of a_param, its derivative
  int* counter;
  int chains, slabs, total;
  uint32_t inv_chains, inv_slabs;
};

// JOIN (gated forward, float32): y leaves as y * gelu(in[3]), the join of the
// recurrent block's two branches (recurrentgemma/torch/modules.py:627-628, 644).
template <typename T, int MODE, int KL, bool JOIN, bool DEAL>
__global__ void __launch_bounds__(kThreads)
scan_tiles_kernel(ScanTileArgs p, DealArgs d) {
  static_assert(!JOIN || (MODE == kFwdGated && sizeof(T) == 4), "");
  using V = Vec<T>;
  using Lds = TileLds<T>;
  constexpr int N = V::n;
  constexpr int CH = Lds::channels;
  constexpr int NS = streams_of(MODE);
  constexpr bool kBwd = MODE == kBwdPlain || MODE == kBwdGated;
  constexpr bool kGated = MODE == kFwdGated || MODE == kBwdGated;
  // (both types: the hardware's exp2, reciprocal and square root; float32 1 - a^2
  // without the cancellation and sigmoids without the exponent's rounding)
  constexpr bool kFast = sizeof(T) == 2;
  constexpr bool kBias = kGated && !kFast;
  constexpr int kSegs = kThreads / CH;    // scanning threads of a channel
  constexpr int kPer = kGroups / kSegs;   // pairs each of them takes
  constexpr int kSegLane = 64 / kSegs;    // lanes between neighbours
  extern __shared__ __align__(16) unsigned char lds_raw[];
  Lds& lds = *reinterpret_cast<Lds*>(lds_raw);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_len = p.T;
  const int oct = lane % kLanes, q = lane / kLanes;
  const int group = wave * (64 / kLanes) + q;
  const uint32_t row_bytes = (uint32_t)p.W * sizeof(T);
  const uint32_t seq_bytes = (uint32_t)T_len * row_bytes;  // < 2^31 (launcher)
  // which of the streams is y (read one row before the token): backward only
  constexpr int kY = MODE == kBwdPlain ? 2 : 4;

  // Blocks of KL tokens in the order of the recurrence.
  const int blocks = (T_len + KL - 1) / KL;
  const int steps = (blocks + kGroups - 1) / kGroups;

  // A step of a slab of channels.
  struct Place {
    int b, c0, step;
    bool any;
  };
  // (dealt out: scalar divisions, an inverse gives the quotient or one less)
  auto quotient = [](uint32_t n, uint32_t by, uint32_t inverse, uint32_t& rest) {
    uint32_t k = (uint32_t)(((uint64_t)n * inverse) >> 32);
    rest = n - k * by;
    k += rest >= by ? 1u : 0u;
    rest -= rest >= by ? by : 0u;
    return k;
  };
  auto place_of = [&](int ticket) {
    Place z;
    z.any = ticket < d.total;
    uint32_t chain, slab;
    z.step = (int)quotient(z.any ? (uint32_t)ticket : 0u, (uint32_t)d.chains,
                           d.inv_chains, chain);
    z.b = (int)quotient(chain, (uint32_t)d.slabs, d.inv_slabs, slab);
    z.c0 = (int)slab * CH;
    return z;
  };
  auto place_at = [&](int k) {  // of this workgroup's k-th ticket
    return place_of(__builtin_amdgcn_readfirstlane(lds.ticket[k & 3]));
  };
  auto take = [&]() { return atomicAdd(d.counter, 1); };
  Place now, ahead;
  int asked = 0;  // (thread 0) the ticket after `ahead`'s
  if (DEAL) {
    if (tid == 0) {
      const int first = take(), second = take();
      asked = take();
      lds.ticket[0] = first;
      lds.ticket[1] = second;
    }
    __syncthreads();
    now = place_at(0);
    ahead = place_at(1);
  } else {
    // Workgroups go to the eight XCDs in turn: neighbouring slabs of channels,
    // which share cache lines where W is no multiple of a slab, to one of them.
    int block = blockIdx.x;
    const int per_xcd = (int)gridDim.x / 8;
    if (block < 8 * per_xcd) block = (block & 7) * per_xcd + (block >> 3);
    const int slabs = (p.W + CH - 1) / CH;
    now.b = block / slabs;
    now.c0 = (block - now.b * slabs) * CH;
    now.step = 0;
    now.any = true;
    ahead = now;
    ahead.step = 1;
  }
  // this lane's byte offset in a place's rows, which start at its slab (W % N == 0:
  // all of the vector or nothing)
  auto lane_off = [&](const Place& z) {
    return z.c0 + oct * N < p.W ? (uint32_t)(oct * N * sizeof(T)) : kBufferOutOfRange;
  };
  auto rows_of = [&](const void* base, const Place& z) {
    const uint32_t before = (uint32_t)z.c0 * sizeof(T);
    return make_rsrc((const char*)base + (int64_t)z.b * seq_bytes + before,
                     z.any ? seq_bytes - before : 0u);
  };
  auto first_token = [&](int step, int g) {
    const int o = step * kGroups + g;
    return (kBwd ? blocks - 1 - o : o) * KL;  // (may lie before or past the row)
  };
  // Rows in registers.  What step 1 wants of the backward forms (dy and the
  // coefficient's stream) and both streams of the plain forward are asked for
  // a step ahead (`next`), the rest at the top of their own step: they are
  // used behind the scan.  The gated forward's rows are consumed in step 1 and
  // reloaded there.
  u32x4 raw[NS][KL];
  constexpr bool kReload = MODE == kFwdGated;
  constexpr int kCoef = MODE == kBwdGated ? 3 : 1;
  auto is_early = [](int s) {
    return MODE == kFwdPlain || s == 0 || (kBwd && s == kCoef);
  };
  u32x4 next[kReload ? 1 : 2][KL];
  // (dealt out: this step's streams and, those that are asked for a step ahead, the
  // next one's)
  __amdgpu_buffer_rsrc_t rs[NS], rs_ahead[NS];
  uint32_t off_now = lane_off(now), off_ahead = off_now;
#pragma unroll
  for (int s = 0; s < NS; ++s) rs[s] = rs_ahead[s] = rows_of(p.in[s], now);
  auto look_ahead = [&]() __attribute__((always_inline)) {
    if (DEAL) {
      off_ahead = lane_off(ahead);
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (kReload || is_early(s)) rs_ahead[s] = rows_of(p.in[s], ahead);
    }
  };
  auto fetch_from = [&](const __amdgpu_buffer_rsrc_t (&from)[NS], uint32_t off, int s,
                        int t0, int i) __attribute__((always_inline)) {
    const int t = kBwd && s == kY ? t0 + i - 1 : t0 + i;
    // (a row before or past the sequence falls outside the descriptor)
    return __builtin_amdgcn_raw_buffer_load_b128(
        from[s],
        off != kBufferOutOfRange ? off + (uint32_t)t * row_bytes : kBufferOutOfRange,
        0, 0);
  };
  auto fetch = [&](int s, int t0, int i) __attribute__((always_inline)) {
    return fetch_from(rs, off_now, s, t0, i);
  };
  auto fetch_ahead = [&](int s, int t0, int i) __attribute__((always_inline)) {
    return DEAL ? fetch_from(rs_ahead, off_ahead, s, t0, i)
                : fetch_from(rs, off_now, s, t0, i);
  };
  // Document starts of the wave's 8 KL tokens, one token per lane.  (Loads of every
  // kind of flag, those that it is not out of range: a branch per kind, or a comparison
  // here, makes the wave wait for them, and for the rows asked for before, at once.
  // us with such waits / without: float32 plain forward B4 T1024 W2560 34.6 / 33.4;
  // prefill, gated forward included, 8 x 2048 472 / 469, 16 x 300 158 / 155, 4 x 700
  // 93.9 / 92.4, but 3 x 1001 89.8 / 91.5; gated backward B4 T1024 98.1 / 95.4, bf16
  // B4 T2048 117.4 / 115.9.)
  const bool flag_bytes = p.flag_kind == kSegMaskU8;
  const uint32_t flag_size = flag_bytes ? 1u : p.flag_kind == kSegI32 ? 4u : 8u;
  uint32_t flag_lo = 0, flag_hi = 0, flag_byte = 0;
  bool flag_in = false;
  auto load_flags = [&](const Place& z) {
    const int lo = first_token(z.step, kBwd ? wave * 8 + 7 : wave * 8);
    const int t = lo + lane;
    flag_in = lane < 8 * KL && t >= 0 && t < T_len;
    const uint32_t row = (uint32_t)T_len * flag_size;  // < 2^31 (scan_tiles_take)
    const __amdgpu_buffer_rsrc_t r =
        make_rsrc((const char*)p.flags + (int64_t)z.b * row, row);
    const uint32_t at = flag_in ? (uint32_t)t * flag_size : kBufferOutOfRange;
    flag_byte = __builtin_amdgcn_raw_buffer_load_b8(
        r, flag_bytes ? at : kBufferOutOfRange, 0, 0);
    flag_lo = __builtin_amdgcn_raw_buffer_load_b32(
        r, flag_bytes ? kBufferOutOfRange : at, 0, 0);
    flag_hi = __builtin_amdgcn_raw_buffer_load_b32(
        r, flag_size == 8u ? at + 4u : kBufferOutOfRange, 0, 0);
  };
  auto is_start = [&]() {
    return flag_in && (flag_bytes ? flag_byte != 0u : (flag_lo | flag_hi) == 0u);
  };

  // softplus of a_param, log2 a = -8 log2(e) sp sigmoid(.): read from LDS
  // twice a step (no registers to keep it in)
  auto channel_value = [&](const void* v, int ch) {
    return ch < p.W ? load_scalar((const T*)v + ch) : 0.0f;
  };
  // (thread ch < CH) its channel's values of a place, asked for and laid into LDS
  float soft[2] = {0.0f, 0.0f}, biases[2] = {0.0f, 0.0f};
  auto ask_channel = [&](const Place& z) __attribute__((always_inline)) {
    if (kGated && tid < CH) {
      const int ch = z.c0 + tid;
      if (DEAL) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
          soft[g] = ch < p.W ? d.soft[(int64_t)g * p.W + ch] : 0.0f;
      } else {
        soft[0] = softplus_precise(channel_value(p.a_param, ch));
      }
      if (kBias) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
          biases[g] = p.bias[g] ? channel_value(p.bias[g], ch) : 0.0f;
      }
    }
  };
  auto lay_channel = [&](const Place& z, int k) __attribute__((always_inline)) {
    if (kGated && tid < CH) {
      lds.sp[k & 1][tid] = soft[0];
      if (DEAL) lds.slope[k & 1][tid] = soft[1];
      if (kBias) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          lds.bias[k & 1][g][tid] = biases[g];
          if (MODE == kFwdGated && p.bias_out && z.any && z.b == 0 && z.step == 0 &&
              z.c0 + tid < p.W)
            p.bias_out[(int64_t)g * p.W + z.c0 + tid] = biases[g];
        }
      }
    }
  };
  if (kGated) {
    ask_channel(now);
    lay_channel(now, 0);
    __syncthreads();
  }
  auto read_row = [&](const float* row, float (&v)[N]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      const f32x4 r = *reinterpret_cast<const f32x4*>(row + oct * N + e);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[e + k] = r[k];
    }
  };
  auto read_sp = [&](int k, float (&sp)[N]) __attribute__((always_inline)) {
    read_row(lds.sp[DEAL ? k & 1 : 0], sp);
  };
  // a gate's pre-activations (0: input, 1: recurrence), the bias included
  auto add_bias = [&](int k, int g, float (&v)[N]) __attribute__((always_inline)) {
    if constexpr (kBias) {
      float b_[N];
      read_row(lds.bias[DEAL ? k & 1 : 0][g], b_);
#pragma unroll
      for (int e = 0; e < N; ++e) v[e] += b_[e];
    }
  };
  auto sigmoid_of = [](float v) __attribute__((always_inline)) {
    return kFast ? sigmoid_fast(v) : sigmoid_f32(v);
  };
  // 1 - a^2 with a = 2^q
  auto rest_of = [](float q, float a) __attribute__((always_inline)) {
    return kFast ? __builtin_fmaf(-a, a, 1.0f) : one_minus_square(q, a);
  };

  // The scanning thread's channel and its state before the step.
  const int seg = lane / kSegLane;
  const int scan_ch = wave * kSegLane + lane % kSegLane;
  auto initial = [&](const Place& z) {
    return p.init && z.c0 + scan_ch < p.W ? p.init[(int64_t)z.b * p.W + z.c0 + scan_ch]
                                          : 0.0f;
  };
  float carry = DEAL ? 0.0f : initial(now);

  float lam_acc[MODE == kBwdGated ? N : 1];
  // float32: also the sums of the gates' gradients (bf16 has no registers for
  // them, and its weight gradients' kernel forms them)
  constexpr bool kBiasGrads = MODE == kBwdGated && kBias;
  float bias_acc[2][kBiasGrads ? N : 1];
  // What a row's (dealt out: a block's) tokens make of the sums over tokens.
  auto zero_sums = [&]() __attribute__((always_inline)) {
    if (MODE == kBwdGated) {
#pragma unroll
      for (int e = 0; e < N; ++e) lam_acc[e] = 0.0f;
    }
    if (kBiasGrads) {
#pragma unroll
      for (int e = 0; e < N; ++e) bias_acc[0][e] = bias_acc[1][e] = 0.0f;
    }
  };
  auto write_sums = [&](const Place& z, int k) __attribute__((always_inline)) {
    if constexpr (MODE == kBwdGated) {
      // over the groups in order
      auto total = [&](const float (&v)[N]) __attribute__((always_inline)) {
        lds_barrier();
#pragma unroll
        for (int e = 0; e < N; e += 4)
          *reinterpret_cast<f32x4*>(&lds.in[group][oct * N + e]) =
              f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]};
        lds_barrier();
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < kPer; ++i) sum += lds.in[seg * kPer + i][scan_ch];
#pragma unroll
        for (int d_ = 1; d_ < kSegs; d_ *= 2) sum += __shfl_xor(sum, d_ * kSegLane);
        return sum;
      };
      const bool writes = seg == 0 && z.c0 + scan_ch < p.W;
      const int64_t rows = DEAL ? (int64_t)p.B * steps : p.B;
      const int64_t row = DEAL ? (int64_t)z.b * steps + z.step : z.b;
      const int64_t at = row * p.W + z.c0 + scan_ch;
      const float lam = total(lam_acc);
      if (writes)
        p.dlam[at] = lam * (DEAL ? lds.slope[k & 1][scan_ch]
                                 : sigmoid_precise(channel_value(p.a_param,
                                                                 z.c0 + scan_ch)));
      if constexpr (kBiasGrads) {
        if (p.dbias != nullptr) {
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            const float sum = total(bias_acc[g]);
            if (writes) p.dbias[(int64_t)g * rows * p.W + at] = sum;
          }
        }
      }
    }
  };

  load_flags(now);
  {
    const int t0 = first_token(now.step, group);
#pragma unroll
    for (int i = 0; i < KL; ++i)
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (kReload || is_early(s)) raw[s][i] = fetch(s, t0, i);
  }
  // (a row's last step apart: only it can hold the row's end, and undealt nothing
  // comes behind it)
  auto one_step = [&](int k, const Place& now, const Place& ahead,
                      auto LAST) __attribute__((always_inline)) {
    constexpr bool last = decltype(LAST)::value;
    constexpr bool more = DEAL || !last;
    const int t0 = first_token(now.step, group);
    const int next_t0 = first_token(ahead.step, group);
    const int c = now.c0 + oct * N;
    const uint32_t c_off = off_now;
    const bool c_ok = c_off != kBufferOutOfRange;
    if (DEAL) {
      zero_sums();
      ask_channel(ahead);
    }
    if (!kReload) {
#pragma unroll
      for (int j = 0; j < KL; ++j) {
        const int i = kBwd ? KL - 1 - j : j;
#pragma unroll
        for (int s = 0; s < NS; ++s)
          if (!is_early(s)) raw[s][i] = fetch(s, t0, i);
      }
    }
    uint32_t starts;
    {
      const uint64_t mask = __ballot(is_start());
      starts = (uint32_t)(mask >> ((kBwd ? 7 - q : q) * KL)) & ((1u << KL) - 1u);
      if (MODE == kFwdGated && p.starts_out && now.c0 == 0 && flag_in)
        p.starts_out[(int64_t)now.b * T_len + first_token(now.step, wave * 8) + lane] =
            is_start();
    }
    if (more) {
      load_flags(ahead);
      // The plain backward does wait for what it has asked for so far before it asks
      // for the next step's rows.  Forward and backward of B4 T2048 W2560 bf16 with the
      // rows in memory: 91.2 us, without this wait 91.7 (in the last-level cache 64.5
      // and 63.8; both kernels waiting, as they did, 92.2 and 65.8).
      if (MODE == kBwdPlain && !DEAL)
        asm volatile("" : "+v"(flag_byte), "+v"(flag_lo), "+v"(flag_hi));
      if (!kReload) {
#pragma unroll
        for (int j = 0; j < KL; ++j) {
          const int i = kBwd ? KL - 1 - j : j;
          next[0][i] = fetch_ahead(0, next_t0, i);
          next[kReload ? 0 : 1][i] = fetch_ahead(kCoef, next_t0, i);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- 1: this lane's tokens as (P, H) ------------------------------------
    // Kept for the replay: the gated forms' coefficients (the plain ones' are
    // the rows themselves), the forward's scaled inputs, and the float32
    // backward's recurrence gates (bf16 has no registers for them, and its
    // sigmoid is six instructions).
    constexpr bool kKeepGate = MODE == kBwdGated && !kFast;
    float coef[kGated ? KL : 1][N];
    float kept[MODE == kFwdGated || kKeepGate ? KL : 1][N];
    float P[N], H[N], sp[N];
    if (kGated) read_sp(k, sp);
#pragma unroll
    for (int e = 0; e < N; ++e) {
      P[e] = 1.0f;
      H[e] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < KL; ++j) {
      const int i = kBwd ? KL - 1 - j : j;
      const bool start = (starts >> i) & 1u;
      const bool behind = kBwd && t0 + i >= T_len;  // identity
      float first[N];
      V::unpack(raw[0][i], first);
      float cf[N];  // a'
      if constexpr (!kGated) {
        V::unpack(raw[1][i], cf);
      } else {
        float ga[N];
        V::unpack(raw[MODE == kFwdGated ? 2 : 3][i], ga);
        add_bias(k, 1, ga);
        float gx[N];
        if (MODE == kFwdGated) {
          V::unpack(raw[1][i], gx);
          add_bias(k, 0, gx);
        }
#pragma unroll
        for (int e = 0; e < N; ++e) {
          const float gate_a = sigmoid_of(ga[e]);
          const float log2_a = gate_a * ((-8.0f * kLog2e) * sp[e]);
          coef[i][e] = __builtin_amdgcn_exp2f(log2_a);
          cf[e] = coef[i][e];
          if constexpr (kKeepGate) kept[i][e] = gate_a;
          if constexpr (MODE == kFwdGated) {
            const float gate_x = sigmoid_of(gx[e]);
            const float m = choose(
                start, 1.0f, __builtin_amdgcn_sqrtf(rest_of(log2_a, coef[i][e])));
            first[e] = (first[e] * gate_x) * m;
            kept[i][e] = first[e];
          }
        }
      }
#pragma unroll
      for (int e = 0; e < N; ++e) {
        cf[e] = choose(start, 0.0f, kBwd ? choose(behind, 1.0f, cf[e]) : cf[e]);
        if (MODE == kFwdGated) coef[i][e] = cf[e];
        H[e] = kBwd ? cf[e] * (H[e] + first[e])
                    : __builtin_fmaf(cf[e], H[e], first[e]);
        P[e] *= cf[e];
      }
      if (kReload && more) {
#pragma unroll
        for (int s = 0; s < NS; ++s) raw[s][i] = fetch_ahead(s, next_t0, i);
      }
    }
#pragma unroll
    for (int e = 0; e < N; e += 2) {
      // (rows are padded by 8 bytes: 8-byte stores)
      *reinterpret_cast<f32x2*>(&lds.pair[group][2 * (oct * N + e)]) =
          f32x2{P[e], H[e]};
      *reinterpret_cast<f32x2*>(&lds.pair[group][2 * (oct * N + e) + 2]) =
          f32x2{P[e + 1], H[e + 1]};
    }
    lds_barrier();
    if (DEAL) {
      if (tid == 0) {  // (asked for a step ago, there by now)
        lds.ticket[(k + 2) & 3] = asked;
        asked = take();
      }
      lay_channel(ahead, k + 1);
    }

    u32x4 branch[JOIN ? KL : 1];
    if constexpr (JOIN) {
      const __amdgpu_buffer_rsrc_t rg = rows_of(p.in[3], now);
#pragma unroll
      for (int i = 0; i < KL; ++i)
        branch[i] = __builtin_amdgcn_raw_buffer_load_b128(
            rg, c_ok ? c_off + (uint32_t)(t0 + i) * row_bytes : kBufferOutOfRange,
            0, 0);
    }

    // ---- 2: scan over the groups ---------------------------------------------
    {
      // (dealt out) the state behind the step before, from whoever had it: number
      // and value
      uint64_t* words = nullptr;
      uint64_t word = 0;
      bool there = false;
      auto poll = [&]() __attribute__((always_inline)) {
        word = (uint64_t)(uint32_t)now.step << 32;
        if (there)
          word = __hip_atomic_load(words + (int64_t)((now.step + 1) & 1) * p.W,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      if (DEAL) {
        words = d.words + ((int64_t)now.b * 2) * p.W + now.c0 + scan_ch;
        there = now.c0 + scan_ch < p.W;
        if (now.step > 0) poll();
      }
      f32x2 v[kPer];
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        v[i] = *reinterpret_cast<const f32x2*>(
            &lds.pair[seg * kPer + i][2 * scan_ch]);
      float sp_ = 1.0f, sh = 0.0f;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        sh = __builtin_fmaf(v[i][0], sh, v[i][1]);
        sp_ *= v[i][0];
      }
#pragma unroll
      for (int d = 1; d < kSegs; d *= 2) {
        const float pp = __shfl_up(sp_, d * kSegLane);
        const float ph = __shfl_up(sh, d * kSegLane);
        if (seg >= d) {
          sh = __builtin_fmaf(sp_, ph, sh);
          sp_ *= pp;
        }
      }
      float ep = __shfl_up(sp_, kSegLane), eh = __shfl_up(sh, kSegLane);
      if (seg == 0) {
        ep = 1.0f;
        eh = 0.0f;
      }
      if constexpr (DEAL) {
        if (now.step == 0) {
          carry = initial(now);
        } else {
          for (int polls = 0; !__all((uint32_t)(word >> 32) == (uint32_t)now.step);
               ++polls) {
            if (polls == kMaxStatePolls) {
              word = kNoState;
              break;
            }
            poll();
          }
          carry = __uint_as_float((uint32_t)word);
        }
        // this step's to whoever has the next
        if (seg == kSegs - 1 && there && now.step + 1 < steps)
          __hip_atomic_store(
              words + (int64_t)(now.step & 1) * p.W,
              ((uint64_t)(uint32_t)(now.step + 1) << 32) |
                  __float_as_uint(__builtin_fmaf(sp_, carry, sh)),
              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      float s = __builtin_fmaf(ep, carry, eh);
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        lds.in[seg * kPer + i][scan_ch] = s;
        s = __builtin_fmaf(v[i][0], s, v[i][1]);
      }
      if (!DEAL) carry = __shfl(s, (kSegs - 1) * kSegLane + lane % kSegLane);
    }
    lds_barrier();

    // ---- 3: replay ------------------------------------------------------------
    if (MODE == kBwdGated) {
      asm volatile("" ::: "memory");
      read_sp(k, sp);
    }
    float st[N];  // h, or the u that comes in from behind
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(&lds.in[group][oct * N + e]);
#pragma unroll
      for (int k = 0; k < 4; ++k) st[e + k] = v[k];
    }
#pragma unroll
    for (int j = 0; j < KL; ++j) {
      const int i = kBwd ? KL - 1 - j : j;
      const int t = t0 + i;
      const bool start = (starts >> i) & 1u;
      const bool inside = t >= 0 && t < T_len;
      const uint32_t at = c_ok && inside
                              ? c_off + (uint32_t)t * row_bytes
                              : kBufferOutOfRange;
      auto store = [&](int o, u32x4 v) {
        buffer_store_16(v, rows_of(p.out[o], now), at, 0);
      };
      // (out of the compiler's sight: it would keep what it unpacked in step 1
      // in registers instead of the packed rows)
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (!kReload) asm volatile("" : "+v"(raw[s][i]));
      float in0[N], cf[N];
      if (!kReload) V::unpack(raw[0][i], in0);
      if constexpr (!kGated) {
        V::unpack(raw[1][i], cf);
#pragma unroll
        for (int e = 0; e < N; ++e)
          cf[e] = choose(start, 0.0f,
                         kBwd ? choose(t >= T_len, 1.0f, cf[e]) : cf[e]);
      }
      if constexpr (!kBwd) {
#pragma unroll
        for (int e = 0; e < N; ++e)
          st[e] = kGated ? __builtin_fmaf(coef[kGated ? i : 0][e], st[e], kept[kGated ? i : 0][e])
                         : __builtin_fmaf(cf[e], st[e], in0[e]);
        float y[N];
#pragma unroll
        for (int e = 0; e < N; ++e)
          y[e] = JOIN ? gelu_mul_f32(st[e], __uint_as_float(branch[JOIN ? i : 0][e & 3]))
                      : st[e];
        store(0, V::pack(y));
        if (last && p.last && t == T_len - 1 && c_ok) {
#pragma unroll
          for (int e = 0; e < N; ++e) p.last[(int64_t)now.b * p.W + c + e] = st[e];
        }
      } else {
        float hp[N];
        V::unpack(raw[kY][i], hp);
        if (i == 0 && t == 0) {  // (t0 is a multiple of KL)
          // h_{-1} in the activation dtype, 16 bytes a load and one wait
          const __amdgpu_buffer_rsrc_t rh =
              make_rsrc(p.h0 + (int64_t)now.b * p.W, p.h0 ? (uint32_t)p.W * 4u : 0u);
          u32x4 h0[N / 4];
#pragma unroll
          for (int e = 0; e < N; e += 4)
            h0[e / 4] = __builtin_amdgcn_raw_buffer_load_b128(
                rh, c_ok ? 4u * (uint32_t)(c + e) : kBufferOutOfRange, 0, 0);
#pragma unroll
          for (int e = 0; e < N; ++e)
            hp[e] = round_act<T>(__uint_as_float(h0[e / 4][e & 3]));
        }
        float g[N];
#pragma unroll
        for (int e = 0; e < N; ++e) g[e] = in0[e] + st[e];
        if constexpr (MODE == kBwdPlain) {
#pragma unroll
          for (int e = 0; e < N; ++e) st[e] = cf[e] * g[e];
          store(0, V::pack(g));
          float da[N];
#pragma unroll
          for (int e = 0; e < N; ++e) da[e] = choose(start, 0.0f, g[e] * hp[e]);
          store(1, V::pack(da));
        } else {
          float x[N], px[N], pa[N], dx[N], dgx[N], dga[N];
          if (!kKeepGate) V::unpack(raw[3][i], pa);
          V::unpack(raw[1][i], x);
          V::unpack(raw[2][i], px);
          add_bias(k, 0, px);
#pragma unroll
          for (int e = 0; e < N; ++e) {
            const float a = coef[i][e];
            const float gate_a = kKeepGate ? kept[kKeepGate ? i : 0][e] : sigmoid_of(pa[e]);
            const float c_t =
                choose(start, 0.0f, choose(t >= T_len, 1.0f, a));
            st[e] = c_t * g[e];
            const float gr = round_act<T>(g[e]);  // the gradient of xn as a tensor
            const float gate_x = sigmoid_of(px[e]);
            const float om =
                kFast ? 1.0f - a * a
                      : one_minus_square(gate_a * ((-8.0f * kLog2e) * sp[e]), a);
            const float a2 = a * a;
            const float m = choose(start, 1.0f, __builtin_amdgcn_sqrtf(om));
            const float d_gated = gr * m;
            const float d_m = gr * (x[e] * gate_x);
            const float clipped = fmaxf(4.0f * om, 1e-6f);
            const float d_om = d_m * __builtin_amdgcn_rsqf(clipped);
            const float d_log_a = choose(start || !inside, 0.0f,
                                         (gr * hp[e]) * a - 2.0f * a2 * d_om);
            dx[e] = d_gated * gate_x;
            dgx[e] = (d_gated * x[e]) * (gate_x * (1.0f - gate_x));
            dga[e] = (-8.0f * sp[e]) * d_log_a * (gate_a * (1.0f - gate_a));
            lam_acc[e] = __builtin_fmaf(-8.0f * gate_a, d_log_a, lam_acc[e]);
            if constexpr (kBiasGrads) {  // (zeros behind the row's end)
              bias_acc[0][e] += dgx[e];
              bias_acc[1][e] += dga[e];
            }
          }
          store(0, V::pack(dx));
          store(1, V::pack(dgx));
          store(2, V::pack(dga));
        }
        if (i == 0 && p.last && t == 0 && c_ok) {  // dh0
#pragma unroll
          for (int e = 0; e < N; ++e) p.last[(int64_t)now.b * p.W + c + e] = st[e];
        }
      }
    }
    if (more && !kReload) {
#pragma unroll
      for (int i = 0; i < KL; ++i) {
        raw[0][i] = next[0][i];
        raw[kCoef][i] = next[kReload ? 0 : 1][i];
      }
    }
  };
  if constexpr (DEAL) {
    look_ahead();
    for (int k = 0; now.any; ++k) {
      if (kBwd || now.step + 1 < steps) {
        one_step(k, now, ahead, std::false_type{});
      } else {
        one_step(k, now, ahead, std::true_type{});
      }
      write_sums(now, k);
      now = ahead;
      off_now = off_ahead;
#pragma unroll
      for (int s = 0; s < NS; ++s)
        rs[s] = kReload || is_early(s) ? rs_ahead[s] : rows_of(p.in[s], now);
      ahead = place_at(k + 2);
      look_ahead();
    }
  } else {
    zero_sums();
    for (; now.step + 1 < steps; ++now.step, ++ahead.step)
      one_step(0, now, ahead, std::false_type{});
    one_step(0, now, ahead, std::true_type{});
    write_sums(now, 0);
  }
}

// Before a dealt launch: no state valid, no ticket taken; softplus of a_param and its
// derivative.
template <typename T>
__global__ void __launch_bounds__(256)
deal_begin_kernel(u32x4* words, int64_t n, const T* a_param, float* soft, int W) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) words[i] = u32x4{0, 0, 0, 0};
  if (a_param != nullptr && i < W) {
    const float v = load_scalar(a_param + i);
    soft[i] = softplus_precise(v);
    soft[W + i] = sigmoid_precise(v);
  }
}

// Tokens of a step.
int step_tokens(int mode) { return (mode == kFwdPlain ? 8 : 4) * kGroups; }

template <typename T, int MODE, int KL, bool JOIN, bool DEAL>
hipError_t launch_form(const ScanTileArgs& a, hipStream_t s) {
  constexpr int lds = sizeof(TileLds<T>);
  static OncePerDevice once;
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)scan_tiles_kernel<T, MODE, KL, JOIN, DEAL>, lds);
  if (e != hipSuccess) return e;
  const int slabs = (a.W + TileLds<T>::channels - 1) / TileLds<T>::channels;
  int64_t blocks = (int64_t)a.B * slabs;
  if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
  DealArgs d{};
  if (DEAL) {
    const int64_t steps = scan_tiles_steps(a.T, MODE);
    if (steps * blocks > (1 << 30)) return hipErrorInvalidValue;
    d.words = (uint64_t*)a.deal;
    const int64_t words = (int64_t)a.B * 2 * a.W;
    d.counter = (int*)(d.words + words);  // (16 bytes of its own)
    d.soft = (float*)(d.counter + 4);
    d.chains = (int)blocks;
    d.slabs = slabs;
    d.inv_chains = 0xffffffffu / (uint32_t)blocks;
    d.inv_slabs = 0xffffffffu / (uint32_t)slabs;
    d.total = (int)(steps * blocks);
    const int64_t items = words / 2 + 1;  // (at least W)
    deal_begin_kernel<T><<<dim3((unsigned)((items + 255) / 256)), 256, 0, s>>>(
        (u32x4*)a.deal, items, (const T*)a.a_param, d.soft, a.W);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    blocks = d.total < 256 ? d.total : 256;
  }
  scan_tiles_kernel<T, MODE, KL, JOIN, DEAL>
      <<<dim3((unsigned)blocks), kThreads, lds, s>>>(a, d);
  return hipGetLastError();
}

template <typename T, int MODE, int KL, bool JOIN = false>
hipError_t launch_as(const ScanTileArgs& a, hipStream_t s) {
  return a.deal ? launch_form<T, MODE, KL, JOIN, true>(a, s)
                : launch_form<T, MODE, KL, JOIN, false>(a, s);
}

}  // namespace

// The gated backward against rg_scan_bwd.hip's: rounds of 256 workgroups by what
// one takes, us.  There: 64 channels a workgroup or, two to a lane, 128, by the
// token; here: steps of 256 tokens.  Both sides as measured (bf16 unless said):
//   B2 T64 W2560 13, here 17, T256 22 / 18, T1024 62 / 52; B8 T64 W2560 21 / 30,
//   T384 54 / 56, T512 69 / 57; B8 W4096 (a full round there, two here) T256 38 /
//   43, T1024 138 / 138, T2048 284 / 329; B16 W4096 T128 43 / 64, T1024 270 / 326,
//   T4096 1118 / 966; B16 T512 W2560 117 / 100; B24 W4096 T384 157 / 187, T1024
//   399 / 365; float32 B2 T64 W2560 14 / 16, T128 19 / 17; B16 W4096 T512 272 /
//   308, T1024 536 / 505; B16 T128 W2560 61 / 75, T256 120 / 97
static bool gated_backward_pays(int B, int T, int W, int dtype, int64_t blocks) {
  const auto rounds = [](int64_t n) { return (float)((n + 255) / 256); };
  const bool two = scan_backward_two_channels(B, W);
  const float one_there = dtype == 0 ? (two ? 10.0f + 0.25f * T : 8.0f + 0.115f * T)
                                     : (two ? 12.0f + 0.105f * T : 10.0f + 0.056f * T);
  const int slabs_there = two ? (W + 127) / 128 : (W + 63) / 64;
  const float there = rounds((int64_t)B * slabs_there) * one_there;
  // (a step behind the second costs by its tokens)
  const float steps = T <= 512 ? (float)((T + 255) / 256) : T / 256.0f;
  const float here = rounds(blocks) * (9.0f + 13.1f * steps);
  // (many or long rows, which that kernel reads twice from memory, take it longer)
  return here < there || T > (blocks <= 1024 ? 2048 : 512);
}

bool scan_tiles_take(int T, int W, int dtype) {
  const int64_t es = dtype == 0 ? 4 : 2;
  return (int64_t)W * es % 16 == 0 &&
         ((int64_t)T + 1024) * W * es < (int64_t)0x7fffffff;
}

bool scan_tiles_serve(int B, int T, int W, int dtype, int mode) {
  const int64_t es = dtype == 0 ? 4 : 2;
  if (!scan_tiles_take(T, W, dtype)) return false;
  // The eight waves of a workgroup walk a slab of channels in steps of 256
  // or 512 tokens, one workgroup per CU: a launch costs a round of the chip per
  // 256 slabs and at least one step, where rg_scan.hip's and rg_scan_bwd.hip's
  // kernels cost by the token.  The lines below are where they meet.
  const int64_t slab = dtype == 0 ? TileLds<float>::channels : TileLds<uint16_t>::channels;
  const int64_t blocks = (int64_t)B * ((W + slab - 1) / slab);
  if (mode == kBwdGated) return gated_backward_pays(B, T, W, dtype, blocks);
  // Both directions of a float32 RG-LRU, which saves four launches beside the
  // kernels' own difference: a whole RGLRU step, us, without and with them: B2 T64
  // W2560 175, 154; B8 W4096 T16 174, 195, T64 188, 175; B16 W2560 T64 252, 259,
  // T128 359, 325; B16 W4096 T128 399, 432, T256 743, 686.
  if (mode == kTilesPairGated)
    return T >= (blocks <= 640 ? 1 : blocks <= 1024 ? 64 : blocks < 2048 ? 100 : 192);
  // The plain backward but for several rounds of short rows (us, B4 T2048 W2560
  // bf16 77 -> 40, B16 T8192 W4096 1555 -> 1104; but B16 T64 W4096 13, here 19;
  // float32 22, here 28).
  if (mode == kBwdPlain)
    return dtype == 0 ? blocks < 800 || T >= 128 : blocks < 512 || T >= 400;
  // The forward ones (B4 T2048 W2560 bf16: plain 52 -> 28, gated 83 -> 44).
  // One or two long rows rg_scan.hip cuts into chunks (bf16 plain: B1 T4096
  // W512 26, here 32, W4096 60, here 41; gated from 4096 tokens on: T8192 105,
  // here 146; float32 plain B1 T8192 W512 60, here 49, gated W2560 T4096 103, here 65,
  // T8192 181, here 152).
  int chunks, t_chunk;
  scan_split_plan(B, T, W, 64, &chunks, &t_chunk);
  if (chunks > 1) {
    const int64_t few = blocks * 64 > 2048 ? blocks * 64 : 2048;
    const int64_t most = mode == kFwdGated ? 4096 : dtype == 0 ? 8192 : few;
    if (T > most && !(mode == kFwdGated && dtype == 0)) return false;
  }
  const bool cached = 3 * es * (int64_t)B * T * W < ((int64_t)256 << 20);
  // Gated: while every slab has a CU of its own; beyond, rows of some length that
  // the last-level cache holds (bf16, projections included: B16 W2560 T64 32, here
  // 40, T256 58, 51, T512 92, 77, T2048 267, 284; B8 W4096 T2048 191, 240; B24 W4096
  // T64 48, 60, T256 96, 84; up to two rounds short rows lose 2 to 6, which the
  // launch that finds the document starts otherwise costs too).  float32: see above.
  if (mode == kFwdGated)
    return dtype == 0 ? blocks < 2048 || cached
                      : blocks <= 256 || (cached && (blocks <= 512 || T >= 128));
  // Plain: while every slab has a CU of its own; beyond, what the last-level
  // cache holds of a few rounds (bf16 B16 T1024 W2560: 62 -> 47, but T300 21,
  // here 22, and B8 T1600 W4096 61, here 71; float32 B8 T500 W2560 30 -> 24, but
  // T180 13, here 14, and B16 T500 W2048 35, here 35).
  if (blocks <= (dtype == 0 ? 512 : 256)) return true;
  return cached && (dtype == 0 ? blocks < 800 && T >= 400 : blocks > 512 && T >= 500);
}

int scan_tiles_steps(int T, int mode) {
  return (T + step_tokens(mode) - 1) / step_tokens(mode);
}

// Dealt out against a slab by the workgroup: us, what a step of a full round and of
// half a round takes (up to 128 slabs leave the memory to each other); dealt, what the
// launches and the first step take, a round of 256 steps, and a step of one row, of
// which the next one waits for its state.  Fitted to 18 shapes a kernel, 1 to 16 rows
// of 1000 to 16000 tokens, 512 to 4096 wide, and within 15 % of them but where the
// planes leave the last-level cache, which slows both alike (slab / dealt: bf16 gated
// backward B1 T2048 W2560 85 / 43, T8192 389 / 112, B4 T2048 118 / 102, B7 T2000
// 206 / 165, but B4 T1024 49 / 58; gated forward B1 T8192 152 / 63, B3 T4096 80 / 73;
// plain backward B1 T8192 130 / 49; float32 gated backward B1 T8192 328 / 163).
static bool dealing_pays(int B, int T, int W, int dtype, int mode) {
  struct Cost {
    float half, full, start, round, row;
  };
  static constexpr Cost kCost[2][4] = {
      // float32: plain forward and backward, gated forward and backward
      {{4.2f, 8.0f, 17.0f, 6.8f, 0.75f}, {3.4f, 6.0f, 17.0f, 5.6f, 0.75f},
       {4.1f, 6.2f, 22.0f, 7.0f, 0.75f}, {7.5f, 15.6f, 22.0f, 13.5f, 0.85f}},
      {{5.2f, 9.0f, 18.0f, 7.6f, 0.75f}, {4.2f, 7.4f, 17.0f, 6.6f, 0.75f},
       {4.8f, 6.8f, 20.0f, 7.6f, 0.75f}, {10.6f, 17.4f, 20.0f, 16.5f, 0.85f}}};
  const int64_t slab = dtype == 0 ? TileLds<float>::channels : TileLds<uint16_t>::channels;
  const int64_t slabs = (int64_t)B * ((W + slab - 1) / slab);
  const int64_t steps = scan_tiles_steps(T, mode);
  if (steps < 2 || steps * slabs > (1 << 30)) return false;
  const Cost& c = kCost[dtype != 0][mode];
  const int64_t rest = slabs % 256;
  const float last =
      rest == 0 ? 0.0f
                : c.half + (c.full - c.half) *
                               sqrtf(fmaxf(0.0f, (float)(rest - 128) / 128.0f));
  const float whole = 2.0f + (float)steps * ((float)(slabs / 256) * c.full + last);
  const float rounds = (float)(steps * slabs) / 256.0f;
  const float dealt = c.start + fmaxf(c.round * rounds, c.row * (float)steps);
  // (its one launch more is time of the host, which short rows are waiting for)
  const bool backward = mode == kBwdPlain || mode == kBwdGated;
  if (whole < (backward ? 55.0f : 30.0f)) return false;
  // (what rg_scan.hip cuts into chunks takes it 0.7 of a slab by the workgroup's time
  // and more: bf16 B1 T8192 W2560 plain 75, gated 100, dealt 38 and 63; B1 T16000 W512
  // 229 and 242, dealt 41 and 65)
  const bool served = scan_tiles_serve(B, T, W, dtype, mode);
  return dealt < (served ? 0.95f : backward ? 0.0f : 0.7f) * whole;
}

size_t scan_tiles_deal_bytes(int B, int T, int W, int dtype, int mode) {
  if (B <= 0 || T <= 0 || W <= 0 || !scan_tiles_take(T, W, dtype) ||
      !dealing_pays(B, T, W, dtype, mode))
    return 0;
  // states, the counter, softplus of a_param and its derivative
  return (size_t)B * 2 * W * 8 + 16 + (((size_t)W * 8 + 15) & ~(size_t)15);
}

hipError_t launch_scan_tiles(const ScanTileArgs& a, int mode, int dtype,
                             hipStream_t s) {
  if (dtype == 0) {
    switch (mode) {
      case kFwdPlain: return launch_as<float, kFwdPlain, 8>(a, s);
      case kBwdPlain: return launch_as<float, kBwdPlain, 4>(a, s);
      case kFwdGated:
        return a.in[3] ? launch_as<float, kFwdGated, 4, true>(a, s)
                       : launch_as<float, kFwdGated, 4>(a, s);
      default: return launch_as<float, kBwdGated, 4>(a, s);
    }
  }
  switch (mode) {
    case kFwdPlain: return launch_as<uint16_t, kFwdPlain, 8>(a, s);
    case kBwdPlain: return launch_as<uint16_t, kBwdPlain, 4>(a, s);
    case kFwdGated: return launch_as<uint16_t, kFwdGated, 4>(a, s);
    default: return launch_as<uint16_t, kBwdGated, 4>(a, s);
  }
}

}  // namespace rg
