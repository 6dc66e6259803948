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
// rounded square would keep few of its digits, -2q (ln 2 + 2q (ln 2)^2 / 2! + ..),
// eight terms of the exponential's series (the ninth is 2e-8 of the first).  With
// it the float32 forms can use the hardware's exp2, reciprocal and square root
// (RG-LRU step B3 T1001 W2560: 254 -> 238 us against expf, sqrtf and divisions)
// and are closer to 64 bits (y 1.9e-7 -> 1.2e-7, its gradients 2.2e-7 .. 4.0e-7
// -> 1.4e-7 .. 2.4e-7, the projections' part of that included).
__device__ __forceinline__ float one_minus_square(float q, float a) {
  constexpr float kSeries[8] = {0.69314718056f,    0.24022650696f,
                                5.5504108665e-2f,  9.6181291076e-3f,
                                1.3333558146e-3f,  1.5403530393e-4f,
                                1.5252733804e-5f,  1.3215486790e-6f};
  const float w = 2.0f * q;
  float s = kSeries[7];
#pragma unroll
  for (int k = 6; k >= 0; --k) s = __builtin_fmaf(s, w, kSeries[k]);
  return w > -0.75f ? -w * s : __builtin_fmaf(-a, a, 1.0f);
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
  float sp[channels];                     // softplus of a_param
  float bias[2][channels];                // float32: of the gate projections
};

// JOIN (gated forward, float32): y leaves as y * gelu(in[3]), the join of the
// recurrent block's two branches (recurrentgemma/torch/modules.py:627-628, 644).
template <typename T, int MODE, int KL, bool JOIN = false>
__global__ void __launch_bounds__(kThreads) scan_tiles_kernel(ScanTileArgs p) {
  static_assert(!JOIN || (MODE == kFwdGated && sizeof(T) == 4), "");
  using V = Vec<T>;
  using Lds = TileLds<T>;
  constexpr int N = V::n;
  constexpr int CH = Lds::channels;
  constexpr int NS = streams_of(MODE);
  constexpr bool kBwd = MODE == kBwdPlain || MODE == kBwdGated;
  constexpr bool kGated = MODE == kFwdGated || MODE == kBwdGated;
  // (both types: the hardware's exp2, reciprocal and square root; float32 forms
  // 1 - a^2 without the cancellation, see below)
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
  // Workgroups go to the eight XCDs in turn: neighbouring slabs of channels,
  // which share cache lines where W is no multiple of a slab, to one of them.
  int block = blockIdx.x;
  {
    const int per_xcd = (int)gridDim.x / 8;
    if (block < 8 * per_xcd) block = (block & 7) * per_xcd + (block >> 3);
  }
  const int slabs = (p.W + CH - 1) / CH;
  const int b = block / slabs;
  const int c0 = (block - b * slabs) * CH;
  const int T_len = p.T;
  const int oct = lane % kLanes, q = lane / kLanes;
  const int group = wave * (64 / kLanes) + q;
  const int c = c0 + oct * N;
  const bool c_ok = c < p.W;  // W % N == 0: all of the vector or nothing

  const uint32_t row_bytes = (uint32_t)p.W * sizeof(T);
  const uint32_t seq_bytes = (uint32_t)T_len * row_bytes;  // < 2^31 (launcher)
  __amdgpu_buffer_rsrc_t rs[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s)
    rs[s] = make_rsrc((const char*)p.in[s] + (int64_t)b * seq_bytes, seq_bytes);
  // which of them is y (read one row before the token): backward only
  constexpr int kY = MODE == kBwdPlain ? 2 : 4;
  const uint32_t c_off = (uint32_t)c * sizeof(T);

  // Blocks of KL tokens in the order of the recurrence.
  const int blocks = (T_len + KL - 1) / KL;
  const int steps = (blocks + kGroups - 1) / kGroups;
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
  auto fetch = [&](int s, int t0, int i) {
    const int t = kBwd && s == kY ? t0 + i - 1 : t0 + i;
    // (a row before or past the sequence falls outside the descriptor)
    return __builtin_amdgcn_raw_buffer_load_b128(
        rs[s], c_ok ? c_off + (uint32_t)t * row_bytes : kBufferOutOfRange, 0, 0);
  };
  // Document starts of the wave's 8 KL tokens, one token per lane.
  uint32_t flag_lo = 1, flag_hi = 0;
  bool flag_in = false;
  auto load_flags = [&](int step) {
    const int lo = first_token(step, kBwd ? wave * 8 + 7 : wave * 8);
    const int t = lo + lane;
    flag_in = lane < 8 * KL && t >= 0 && t < T_len;
    const int64_t at = (int64_t)b * T_len + (flag_in ? t : 0);
    if (p.flag_kind == kSegMaskU8) {
      flag_lo = reinterpret_cast<const uint8_t*>(p.flags)[at] == 0;
      flag_hi = 0;
    } else if (p.flag_kind == kSegI32) {
      flag_lo = reinterpret_cast<const uint32_t*>(p.flags)[at];
      flag_hi = 0;
    } else {
      const u32x2 v = reinterpret_cast<const u32x2*>(p.flags)[at];
      flag_lo = v[0];
      flag_hi = v[1];
    }
  };

  // softplus of a_param, log2 a = -8 log2(e) sp sigmoid(.): read from LDS
  // twice a step (no registers to keep it in)
  auto lambda_of = [&](int ch) {  // a_param of the workgroup's channel ch
    return c0 + ch < p.W ? load_scalar((const T*)p.a_param + c0 + ch) : 0.0f;
  };
  if (kGated) {
    if (tid < CH) {
      lds.sp[tid] = softplus_precise(lambda_of(tid));
      if (kBias) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          lds.bias[g][tid] = p.bias[g] && c0 + tid < p.W
                                 ? load_scalar((const T*)p.bias[g] + c0 + tid)
                                 : 0.0f;
          if (MODE == kFwdGated && p.bias_out && b == 0 && c0 + tid < p.W)
            p.bias_out[(int64_t)g * p.W + c0 + tid] = lds.bias[g][tid];
        }
      }
    }
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
  auto read_sp = [&](float (&sp)[N]) __attribute__((always_inline)) {
    read_row(lds.sp, sp);
  };
  // a gate's pre-activations (0: input, 1: recurrence), the bias included
  auto add_bias = [&](int g, float (&v)[N]) __attribute__((always_inline)) {
    if constexpr (kBias) {
      float b_[N];
      read_row(lds.bias[g], b_);
#pragma unroll
      for (int e = 0; e < N; ++e) v[e] += b_[e];
    }
  };
  // 1 - a^2 with a = 2^q
  auto rest_of = [](float q, float a) __attribute__((always_inline)) {
    return kFast ? __builtin_fmaf(-a, a, 1.0f) : one_minus_square(q, a);
  };

  // The scanning thread's channel and its state before the step.
  const int seg = lane / kSegLane;
  const int scan_ch = wave * kSegLane + lane % kSegLane;
  float carry = 0.0f;
  if (p.init && c0 + scan_ch < p.W)
    carry = p.init[(int64_t)b * p.W + c0 + scan_ch];

  float lam_acc[MODE == kBwdGated ? N : 1];
  // float32: also the sums of the gates' gradients (bf16 has no registers for
  // them, and its weight gradients' kernel forms them)
  constexpr bool kBiasGrads = MODE == kBwdGated && kBias;
  float bias_acc[2][kBiasGrads ? N : 1];
  if (MODE == kBwdGated) {
#pragma unroll
    for (int e = 0; e < N; ++e) lam_acc[e] = 0.0f;
  }
  if (kBiasGrads) {
#pragma unroll
    for (int e = 0; e < N; ++e) bias_acc[0][e] = bias_acc[1][e] = 0.0f;
  }

  load_flags(0);
  {
    const int t0 = first_token(0, group);
#pragma unroll
    for (int i = 0; i < KL; ++i)
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (kReload || is_early(s)) raw[s][i] = fetch(s, t0, i);
  }
  // (the last step apart: only it can hold the row's end)
  auto one_step = [&](int step, auto LAST) __attribute__((always_inline)) {
    constexpr bool more = !decltype(LAST)::value;
    const int t0 = first_token(step, group);
    const int next_t0 = first_token(step + 1, group);
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
      const uint64_t mask = __ballot(flag_in && (flag_lo | flag_hi) == 0u);
      starts = (uint32_t)(mask >> ((kBwd ? 7 - q : q) * KL)) & ((1u << KL) - 1u);
      if (MODE == kFwdGated && p.starts_out && c0 == 0 && flag_in)
        p.starts_out[(int64_t)b * T_len + first_token(step, wave * 8) + lane] =
            (flag_lo | flag_hi) == 0u;
    }
    if (more) {
      load_flags(step + 1);
      if (!kReload) {
#pragma unroll
        for (int j = 0; j < KL; ++j) {
          const int i = kBwd ? KL - 1 - j : j;
          next[0][i] = fetch(0, next_t0, i);
          next[kReload ? 0 : 1][i] = fetch(kCoef, next_t0, i);
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
    if (kGated) read_sp(sp);
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
        add_bias(1, ga);
        float gx[N];
        if (MODE == kFwdGated) {
          V::unpack(raw[1][i], gx);
          add_bias(0, gx);
        }
#pragma unroll
        for (int e = 0; e < N; ++e) {
          const float gate_a = sigmoid_fast(ga[e]);
          const float log2_a = gate_a * ((-8.0f * kLog2e) * sp[e]);
          coef[i][e] = __builtin_amdgcn_exp2f(log2_a);
          cf[e] = coef[i][e];
          if constexpr (kKeepGate) kept[i][e] = gate_a;
          if constexpr (MODE == kFwdGated) {
            const float gate_x = sigmoid_fast(gx[e]);
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
        for (int s = 0; s < NS; ++s) raw[s][i] = fetch(s, next_t0, i);
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

    u32x4 branch[JOIN ? KL : 1];
    if constexpr (JOIN) {
      const __amdgpu_buffer_rsrc_t rg = make_rsrc(
          (const char*)p.in[3] + (int64_t)b * seq_bytes, seq_bytes);
#pragma unroll
      for (int i = 0; i < KL; ++i)
        branch[i] = __builtin_amdgcn_raw_buffer_load_b128(
            rg, c_ok ? c_off + (uint32_t)(t0 + i) * row_bytes : kBufferOutOfRange,
            0, 0);
    }

    // ---- 2: scan over the groups ---------------------------------------------
    {
      f32x2 v[kPer];
#pragma unroll
      for (int k = 0; k < kPer; ++k)
        v[k] = *reinterpret_cast<const f32x2*>(
            &lds.pair[seg * kPer + k][2 * scan_ch]);
      float sp_ = 1.0f, sh = 0.0f;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        sh = __builtin_fmaf(v[k][0], sh, v[k][1]);
        sp_ *= v[k][0];
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
      float s = __builtin_fmaf(ep, carry, eh);
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        lds.in[seg * kPer + k][scan_ch] = s;
        s = __builtin_fmaf(v[k][0], s, v[k][1]);
      }
      carry = __shfl(s, (kSegs - 1) * kSegLane + lane % kSegLane);
    }
    lds_barrier();

    // ---- 3: replay ------------------------------------------------------------
    if (MODE == kBwdGated) {
      asm volatile("" ::: "memory");
      read_sp(sp);
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
        buffer_store_16(v, make_rsrc((char*)p.out[o] + (int64_t)b * seq_bytes,
                                     seq_bytes), at, 0);
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
        if (!more && p.last && t == T_len - 1 && c_ok) {
#pragma unroll
          for (int e = 0; e < N; ++e) p.last[(int64_t)b * p.W + c + e] = st[e];
        }
      } else {
        float hp[N];
        V::unpack(raw[kY][i], hp);
        if (i == 0 && t == 0) {  // (t0 is a multiple of KL)
#pragma unroll
          for (int e = 0; e < N; ++e)  // h_{-1} in the activation dtype
            hp[e] = p.h0 && c_ok ? round_act<T>(p.h0[(int64_t)b * p.W + c + e])
                                 : 0.0f;
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
          add_bias(0, px);
#pragma unroll
          for (int e = 0; e < N; ++e) {
            const float a = coef[i][e];
            const float gate_a = kKeepGate ? kept[kKeepGate ? i : 0][e] : sigmoid_fast(pa[e]);
            const float c_t =
                choose(start, 0.0f, choose(t >= T_len, 1.0f, a));
            st[e] = c_t * g[e];
            const float gr = round_act<T>(g[e]);  // the gradient of xn as a tensor
            const float gate_x = sigmoid_fast(px[e]);
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
          for (int e = 0; e < N; ++e) p.last[(int64_t)b * p.W + c + e] = st[e];
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
  for (int step = 0; step + 1 < steps; ++step) one_step(step, std::false_type{});
  one_step(steps - 1, std::true_type{});

  if constexpr (MODE == kBwdGated) {
    // sums over the row: over the groups in order
    auto total = [&](const float (&v)[N]) __attribute__((always_inline)) {
      __syncthreads();
#pragma unroll
      for (int e = 0; e < N; e += 4)
        *reinterpret_cast<f32x4*>(&lds.in[group][oct * N + e]) =
            f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]};
      __syncthreads();
      float sum = 0.0f;
#pragma unroll
      for (int k = 0; k < kPer; ++k) sum += lds.in[seg * kPer + k][scan_ch];
#pragma unroll
      for (int d = 1; d < kSegs; d *= 2) sum += __shfl_xor(sum, d * kSegLane);
      return sum;
    };
    const bool writes = seg == 0 && c0 + scan_ch < p.W;
    const int64_t at = (int64_t)b * p.W + c0 + scan_ch;
    const float lam = total(lam_acc);
    if (writes) p.dlam[at] = lam * sigmoid_precise(lambda_of(scan_ch));
    if constexpr (kBiasGrads) {
      if (p.dbias != nullptr) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const float sum = total(bias_acc[g]);
          if (writes) p.dbias[(int64_t)g * p.B * p.W + at] = sum;
        }
      }
    }
  }
}

template <typename T, int MODE, int KL, bool JOIN = false>
hipError_t launch_as(const ScanTileArgs& a, hipStream_t s) {
  constexpr int lds = sizeof(TileLds<T>);
  static OncePerDevice once;
  hipError_t e =
      set_max_dynamic_lds(once, (const void*)scan_tiles_kernel<T, MODE, KL, JOIN>,
                          lds);
  if (e != hipSuccess) return e;
  const int64_t blocks =
      (int64_t)a.B * ((a.W + TileLds<T>::channels - 1) / TileLds<T>::channels);
  if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
  scan_tiles_kernel<T, MODE, KL, JOIN>
      <<<dim3((unsigned)blocks), kThreads, lds, s>>>(a);
  return hipGetLastError();
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
  // here 146; float32 plain B1 T8192 W512 60, here 49).
  int chunks, t_chunk;
  scan_split_plan(B, T, W, 64, &chunks, &t_chunk);
  if (chunks > 1) {
    const int64_t few = blocks * 64 > 2048 ? blocks * 64 : 2048;
    const int64_t most = mode == kFwdGated ? 4096 : dtype == 0 ? 8192 : few;
    if (T > most) return false;
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
