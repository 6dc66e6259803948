// Recurrent core of a prefill in one launch (bf16, heads of 128 .. 256
// channels), the form for few (row, head) pairs, for rows of a few tokens and
// for heads narrower than 256: a head's channels are cut into slices of 64,
// and a workgroup of eight waves works on four tiles of 32 tokens at once.
//
// The forms that give a workgroup a whole head walk a row block by block, 2.1
// us per 32 tokens, and fill the chip only from 256 pairs on.  Here a
// workgroup owns 64 output channels of one head (both gates) and a range of
// rows.  A pass takes the next four tiles of 32 tokens of those rows -- four
// tiles of a long row, or tiles of up to four different rows:
//   * conv: each wave convolves a tile of the pass over half of the head's
//     channels (every slice of the head convolves them again: 3.75 vector slots per
//     element and slice, the price of the split) into an LDS tile;
//   * wave (tile, half of the slice) multiplies its 32 tokens by its 32
//     channels of both gates, the weights (2 KS fragments) resident in
//     accumulation registers; the conv of the NEXT pass is issued between the
//     matrix instructions;
//   * gates, then the recurrence: a lane has 16 tokens of one channel; it
//     forms the tile's (prod a, state from zero), the four tiles' pairs meet
//     in LDS, every wave folds the tiles before its own onto the carried state
//     (the scan operator of recurrentgemma/jax/scan.py:161-187), and replays.
// One workgroup barrier per pass: the conv tile and the pairs are double
// buffered.  Arithmetic and roundings are those of rg_prefill_teams.hip except
// for the order in which the float32 state is combined.
//
// What bounds it: vector issue, like the other forms (about 1.6 times their
// slots per element, because of the repeated conv).
//
// Replaces the chain Conv1D.forward -> RGLRU.forward of
// recurrentgemma/torch/modules.py:632-643 (layers.py:447-529, 313-365,
// 140-191) for such shapes.
#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"
#include "rg_weight_frags.h"

namespace rg {
namespace {

#define RG_INLINE __attribute__((always_inline))

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kTile = 32;                     // tokens per tile
constexpr int kTiles = 4;                     // tiles per pass
constexpr int kSlice = 64;                    // channels per workgroup
constexpr int kConvRows = kTile;              // conv rows of a wave: one tile
constexpr int kPatchStride = 80;              // bytes: 32 channels + padding
constexpr int kPatchBytes = 16 * kPatchStride;
constexpr int kARing = 3;

typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) f32x2 lds_f32x2;

// LDS, in bytes: two conv tiles of four times 32 tokens, every matrix wave's
// output patch, the tiles' (prod a, state) pairs twice, conv taps, and the
// biases and inverse decays of the workgroup's channels.
template <int KS>
struct Layout {
  static constexpr int row = (KS * 16 + 8) * 2;
  static constexpr int buffer = kTile * kTiles * row;
  static constexpr int patch = 2 * buffer;
  static constexpr int pairs = patch + kWaves * kPatchBytes;
  static constexpr int pairs_one = kTiles * kSlice * 8;
  static constexpr int taps = pairs + 2 * pairs_one;
  static constexpr int gates = taps + 128 * 32;
  static constexpr int total = gates + kSlice * 16;
  static_assert(total <= 160 * 1024, "LDS of one CU");
};

// (a loop that must be unrolled: the fragment numbers are constants)
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// The 2 KS matrix instructions of a tile; between(ks) is issued behind those of
// k-step ks.
template <int KS, class F>
__device__ __forceinline__ void matrix_tile(lds_byte* const lds3,
                                            const uint32_t a_at, f32x16& acc_x,
                                            f32x16& acc_a, F&& between) {
  auto a_read = [&](int ks) RG_INLINE {
    return *reinterpret_cast<lds_f32x4*>(lds3 + a_at + ks * 32);
  };
  f32x4 a[kARing];
#pragma unroll
  for (int k = 0; k < kARing - 1; ++k) a[k] = a_read(k);
  static_for<0, KS>([&](auto KSTEP) RG_INLINE {
    constexpr int ks = decltype(KSTEP)::value;
    if constexpr (ks + kARing - 1 < KS)
      a[(ks + kARing - 1) % kARing] = a_read(ks + kARing - 1);
    mfma_weight_frag(2 * ks, ks == 0, a[ks % kARing], acc_x);
    mfma_weight_frag(2 * ks + 1, ks == 0, a[ks % kARing], acc_a);
    between(KSTEP);
  });
  // the last matrix results land (19 issue slots)
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc_x), "+v"(acc_a));
}

// One tile of 32 tokens: which row it is in, where, and its document starts.
struct TileAt {
  int row, t0, k_in_row;
  bool any;     // false: past the workgroup's rows
  bool active;  // ... and this wave's channels are channels of the head
  uint32_t starts;
  int tokens;   // of its row (MANY: of the rows that lie in it)
};

// Several whole rows to a tile (MANY): how many, and of the tile's tokens those that
// open a row and those that end one; token i is in the tile's row i * inverse >> 16.
struct RowsOfTile {
  int rows;
  uint32_t opens, ends, inverse;
};

// From a tile's pre-activations (a lane: 16 tokens of one channel, runs of four
// that alternate between the lane halves) to its outputs: gates, the tile as
// (prod a, state from zero), the workgroup's barrier, the fold of the pass's
// four tiles, replay, stores.  c0: this wave's first channel among the workgroup's,
// n0: in the head.  until: how many tiles after the pass's
// first the next row opens (0: that one does), kept up to date here.
template <class L, bool GELU, bool MANY>
__device__ __forceinline__ void gate_and_scan(
    const FusedArgs& p, const RowsOfTile& many, lds_byte* const lds3, const int lane, const int wave,
    const int bw, const int h, const int n0, const int c0, const int tt,
    const int buf, const int tiles_per_row, const TileAt at_tile,
    const f32x16& acc_x, const f32x16& acc_a, float& carry, int& until) {
  const int T = MANY ? at_tile.tokens : p.T;
  const int64_t W = p.W;
  const uint32_t row_bytes = 2u * (uint32_t)p.W;
  const uint32_t seq_bytes = (uint32_t)T * row_bytes;
  const int64_t seq_at =
      (int64_t)at_tile.row * (MANY ? many.rows * p.T : p.T) * row_bytes;
  const int b = at_tile.row, t0 = at_tile.t0, k_in_row = at_tile.k_in_row;
  const bool any = at_tile.any, active = at_tile.active;
  const uint32_t starts = at_tile.starts;
      // (per-lane addresses of the rest of the pass, made again in every pass:
      // kept across the matrix instructions they are registers too many)
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const uint32_t patch_w = L::patch + wave * kPatchBytes +
                               4u * (ln >> 5) * kPatchStride + 2u * (ln & 31);
      const uint32_t patch_r = L::patch + wave * kPatchBytes +
                               (uint32_t)(ln >> 2) * kPatchStride + 16u * (ln & 3);
      const bool ch_valid = n0 + (ln & 31) < bw;
  const bool y_valid = n0 + 8 * (ln & 3) < bw;
      const uint32_t y_lane = (uint32_t)(ln >> 2) * row_bytes +
                              2u * (uint32_t)(h * bw + n0) + 16u * (ln & 3);
      const uint32_t state_off =
          4u * (uint32_t)(h * bw + (n0 + (ln & 31) < bw ? n0 + (ln & 31) : 0));

      // ---- gates ---------------------------------------------------------------
      const bool is_gelu_row = GELU && active;
      u32x4 gate_rows[2];
      if (GELU) {
        const __amdgpu_buffer_rsrc_t rgate =
            make_rsrc((const char*)p.gate_branch + seq_at,
                      is_gelu_row ? seq_bytes : 0);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          gate_rows[j] = __builtin_amdgcn_raw_buffer_load_b128(
              rgate,
              y_valid ? y_lane + (uint32_t)(t0 + 16 * j) * row_bytes
                      : kBufferOutOfRange,
              0, 0);
      }
      const f32x4 per_channel = *reinterpret_cast<lds_f32x4*>(
          lds3 + L::gates + (c0 + (ln & 31)) * 16);
      const float bias_x = per_channel[0], bias_a = per_channel[1];
      const float inv_decay = per_channel[2];
      const uint32_t xc_lane =
          (uint32_t)(tt * kTile + 4 * (ln >> 5)) * L::row + 2u * (uint32_t)(n0 + (ln & 31));
      float av[16], xn[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint16_t xc = *reinterpret_cast<lds_u16*>(
            lds3 + buf * L::buffer + xc_lane + (8 * (e >> 2) + (e & 3)) * L::row);
        xn[e] = bf16_bits_to_f32(xc);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float gx = __builtin_amdgcn_rcpf(
            1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(acc_x[e], -kLog2e, bias_x)));
        av[e] = __builtin_amdgcn_exp2f(gate_exponent(
            __builtin_amdgcn_exp2f(__builtin_fmaf(acc_a[e], -kLog2e, bias_a)),
            inv_decay));
        xn[e] *= gx;
      }
      if (__builtin_expect(starts != 0 || t0 + kTile > T, 0)) {
        // document start: a = 0; past the end of the row: identity.  (The lane
        // half's offset is made here, out of the compiler's sight: it would
        // keep a mask and a bound per element in registers across the loop.)
        int first = (ln >> 5) * 4;
        asm volatile("" : "+v"(first));
        const uint32_t mine = starts >> first;
        const int left = T - t0 - first;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = 8 * (e >> 2) + (e & 3);
          av[e] = (mine >> row) & 1u ? 0.0f : av[e];
          av[e] = row < left ? av[e] : 1.0f;
          xn[e] = row < left ? xn[e] : 0.0f;
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e)
        xn[e] *= __builtin_amdgcn_sqrtf(__builtin_fmaf(-av[e], av[e], 1.0f));
      // MANY: a row that opens in the tile starts from its h0, and is cut from the row
      // before by selection, here and below (runs of four tokens: uniformly).
      // (masks of this lane's tokens, made where they are used: a comparison per
      // element kept across the pass is scalar registers too many)
      uint32_t opens = 0, first_token = 0;
      auto lane_masks = [&]() RG_INLINE {
        if (MANY) {
          first_token = (uint32_t)(ln >> 5) * 4u;
          asm volatile("" : "+v"(first_token));
          opens = many.opens >> first_token;
        }
      };
      if (MANY) {
        if (p.h0) {
          lane_masks();
          const __amdgpu_buffer_rsrc_t rh0 =
              make_rsrc(p.h0 + (int64_t)b * many.rows * W,
                        active ? (uint32_t)(T / p.T) * 2u * row_bytes : 0u);
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const uint32_t row = 8 * (e >> 2) + (e & 3);
            const uint32_t in_tile = (row + first_token) * many.inverse >> 16;
            if (e % 4 == 0) asm volatile("" ::: "memory");
            const float h0 = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           rh0,
                           (opens >> row) & 1u
                               ? in_tile * 2u * row_bytes + state_off
                               : kBufferOutOfRange,
                           0, 0));
            xn[e] = (opens >> row) & 1u ? __builtin_fmaf(av[e], h0, xn[e]) : xn[e];
          }
        }
      }
      auto walk = [&](int e, float state) RG_INLINE {
        const float next = __builtin_fmaf(av[e], state, xn[e]);
        return MANY && ((opens >> (8 * (e >> 2) + (e & 3))) & 1u) ? xn[e] : next;
      };

      // ---- the tile as (prod a, state from zero): runs of four tokens, of the
      //      lower and the upper lanes in turn ---------------------------------
      float run_p[4][2], run_h[4][2];  // [run][lane half]
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        lane_masks();
        float ph = xn[4 * g], pp = av[4 * g];
#pragma unroll
        for (int q = 1; q < 4; ++q) {
          ph = walk(4 * g + q, ph);
          pp *= av[4 * g + q];
        }
        const auto sp = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(pp), __float_as_uint(pp), false, false);
        const auto sh = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(ph), __float_as_uint(ph), false, false);
        run_p[g][0] = __uint_as_float(sp[0]);
        run_p[g][1] = __uint_as_float(sp[1]);
        run_h[g][0] = __uint_as_float(sh[0]);
        run_h[g][1] = __uint_as_float(sh[1]);
      }
      auto walk_run = [&](int g, int s, float state) RG_INLINE {
        const float next = __builtin_fmaf(run_p[g][s], state, run_h[g][s]);
        return MANY && ((many.opens >> (8 * g + 4 * s)) & 15u) ? run_h[g][s] : next;
      };
      float tp = 1.0f, th = 0.0f;
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          th = walk_run(g, s, th);
          tp *= run_p[g][s];
        }
      // a tile that opens its row starts from the row's h0 instead of from zero
      if (k_in_row == 0) {
        const float first =
            !MANY && p.h0 && any && ch_valid
                ? *reinterpret_cast<const float*>(
                      (const char*)(p.h0 + (int64_t)b * W) + state_off)
                : 0.0f;
        th = __builtin_fmaf(tp, first, th);
        if (any) carry = first;
      }
      {
        lds_f32x2* const mine = reinterpret_cast<lds_f32x2*>(
            lds3 + L::pairs + buf * L::pairs_one + (tt * kSlice + c0) * 8);
        if (ln < 32) mine[ln] = f32x2{tp, th};
      }
      lds_barrier();
      // ---- state before this tile, and behind the pass -----------------------
      float hin = carry;
      {
        const lds_f32x2* const all = reinterpret_cast<const lds_f32x2*>(
            lds3 + L::pairs + buf * L::pairs_one + c0 * 8);
        f32x2 v[kTiles];
#pragma unroll
        for (int k = 0; k < kTiles; ++k) v[k] = all[k * kSlice + (ln & 31)];
        float s = carry;
        // rows open in this pass: cut from the row before by selection (a product of
        // zero would let that row's NaN or infinity through; B3 T333 W2560 without the
        // cut 22.61 us, with it 22.64)
        const bool opens = k_in_row == 0;
#pragma unroll
        for (int k = 0; k < kTiles; ++k) {
          if (k == tt && !opens) hin = s;
          const float next = __builtin_fmaf(v[k][0], s, v[k][1]);
          s = k == until ? v[k][1] : next;
          until += k == until ? tiles_per_row : 0;
        }
        until -= kTiles;
        carry = s;
      }
      if (active) {
        // ---- replay -------------------------------------------------------------
        const __amdgpu_buffer_rsrc_t ry =
            make_rsrc((char*)p.y + seq_at, seq_bytes);
        const __amdgpu_buffer_rsrc_t rlast =
            make_rsrc(p.h_last + (MANY ? (int64_t)b * many.rows * W : 0),
                      MANY && p.h_last ? (uint32_t)(T / p.T) * 2u * row_bytes : 0u);
        float s = hin;
        float behind = hin;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float before = s;
          s = walk_run(g, 0, s);
          float hh = ln >= 32 ? s : before;
          s = walk_run(g, 1, s);
          float hv[4];
          lane_masks();
          const uint32_t ends = MANY ? many.ends >> first_token : 0u;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            hh = walk(4 * g + q, hh);
            hv[q] = hh;
            if (MANY) {  // (rows past the last, tokens that end none: dropped)
              const uint32_t row = 8 * g + q;
              const uint32_t in_tile = (row + first_token) * many.inverse >> 16;
              __builtin_amdgcn_raw_buffer_store_b32(
                  __float_as_uint(hh), rlast,
                  ((ends >> row) & 1u) && ch_valid
                      ? in_tile * 2u * row_bytes + state_off
                      : kBufferOutOfRange,
                  0, 0);
            }
          }
          behind = hh;
          const uint32_t y01 = pack_bf16x2(hv[0], hv[1]);
          const uint32_t y23 = pack_bf16x2(hv[2], hv[3]);
          const uint32_t pw = patch_w + (8 * (g & 1)) * kPatchStride;
          asm volatile(
              "ds_write_b16 %0, %1\n\t"
              "ds_write_b16_d16_hi %0, %1 offset:%3\n\t"
              "ds_write_b16 %0, %2 offset:%4\n\t"
              "ds_write_b16_d16_hi %0, %2 offset:%5"
              :
              : "v"(pw), "v"(y01), "v"(y23), "n"(kPatchStride),
                "n"(2 * kPatchStride), "n"(3 * kPatchStride)
              : "memory");
          if (g & 1) {
            u32x4 out = *reinterpret_cast<lds_u32x4*>(lds3 + patch_r);
            asm volatile("" ::: "memory");
            if (GELU) {
#pragma unroll
              for (int k = 0; k < 4; ++k)
                out[k] = gelu_mul_bf16x2(out[k], gate_rows[g >> 1][k]);
            }
            const uint32_t at = (uint32_t)(t0 + 16 * (g >> 1)) * row_bytes;
            buffer_store_16(out, ry, y_valid ? y_lane + at : kBufferOutOfRange, 0);
          }
        }
        // the row's last tile: its end state (identity past the end) -- the
        // upper lanes' last run is the tile's last
        if (!MANY && p.h_last && k_in_row == tiles_per_row - 1 && ln >= 32 &&
            ch_valid)
          *reinterpret_cast<float*>((char*)(p.h_last + (int64_t)b * W) +
                                    state_off) = behind;
      }
}

// The wave's weights, KS k-steps x 2 gates of channels n0 .. n0 + 31 of head h,
// into its accumulation registers; zeros beyond the head.
template <int KS, bool PACKED>
__device__ __forceinline__ void load_weights(const FusedArgs& p, const int lane,
                                             const int bw, const int h,
                                             const int n0) {
  const int n = n0 + (lane & 31);
  const bool n_valid = n < bw;
  if (PACKED) {
    const int nt = (bw + 31) / 32;  // 32-channel groups of a head
    const f32x4* src = reinterpret_cast<const f32x4*>(p.w_packed) +
                       ((int64_t)(h * nt + n0 / 32) * KS * 2) * 64 + lane;
    const bool any = n0 < bw;  // (the last slice's second half may be empty)
#pragma unroll
    for (int f0 = 0; f0 < 2 * KS; f0 += 16) {
      f32x4 w[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        w[i] = f32x4{0, 0, 0, 0};
        if (f0 + i < 2 * KS && any) w[i] = src[(f0 + i) * 64];
      }
      asm volatile("" ::"v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]),
                   "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]),
                   "v"(w[10]), "v"(w[11]), "v"(w[12]), "v"(w[13]), "v"(w[14]),
                   "v"(w[15]));
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (f0 + i < 2 * KS) set_weight_frag(f0 + i, w[i]);
    }
  }
  if (!PACKED) {
#pragma unroll
    for (int f = 0; f < 2 * KS; ++f) {
      const uint16_t* src = (const uint16_t*)p.w[f & 1] +
                            (int64_t)h * bw * bw + (n_valid ? n : 0);
      union {
        uint16_t u[8];
        f32x4 q;
      } w;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = 16 * (f >> 1) + 8 * (lane >> 5) + e;
        w.u[e] = n_valid && k < bw ? src[(int64_t)k * bw] : (uint16_t)0;
      }
      set_weight_frag(f, w.q);
    }
  }
}

// Conv taps of the head's channel pairs, as time pairs (rg_common.h).
template <class L>
__device__ __forceinline__ void fill_taps(const FusedArgs& p,
                                          unsigned char* const lds_raw,
                                          const int tid, const int bw,
                                          const int h) {
  const int64_t W = p.W;
  if (tid < 128) {
    uint32_t u0 = 0, u1 = 0, u2 = 0, u3 = 0x3f803f80u, ub = 0;
    if (p.conv_w != nullptr && tid * 2 < bw) {
      const uint16_t* cw = (const uint16_t*)p.conv_w + h * bw + tid * 2;
      u0 = *reinterpret_cast<const uint32_t*>(cw);
      u1 = *reinterpret_cast<const uint32_t*>(cw + W);
      u2 = *reinterpret_cast<const uint32_t*>(cw + 2 * W);
      u3 = *reinterpret_cast<const uint32_t*>(cw + 3 * W);
      ub = *reinterpret_cast<const uint32_t*>((const uint16_t*)p.conv_b +
                                              h * bw + tid * 2);
    }
    uint32_t w10[2], w32[2];
    pair_up(u0, u1, w10[0], w10[1]);
    pair_up(u2, u3, w32[0], w32[1]);
    u32x4* const tab = reinterpret_cast<u32x4*>(lds_raw + L::taps + tid * 32);
    tab[0] = u32x4{w10[0], w10[1], w32[0], w32[1]};
    tab[1] = u32x4{ub << 16, ub & 0xffff0000u, 0u, 0u};
  }
}
// Biases and inverse decay of channels n0 .. n0 + 31: read back in every pass (kept in
// registers across the matrix instructions they are three too many).
template <class L>
__device__ __forceinline__ void fill_gate_values(const FusedArgs& p,
                                                 unsigned char* const lds_raw,
                                                 const int lane, const int bw,
                                                 const int h, const int n0,
                                                 const int c0) {
  const int n = n0 + (lane & 31);
  if (lane < 32) {
    f32x4 v = {0, 0, 0, 0};
    if (n < bw) {
      v[0] = -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[0])[h * bw + n]);
      v[1] = -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[1])[h * bw + n]);
      v[2] = inverse_decay(
          (-8.0f * kLog2e) *
          softplus_precise(bf16_bits_to_f32(((const uint16_t*)p.a_param)[h * bw + n])));
    }
    *reinterpret_cast<f32x4*>(lds_raw + L::gates + (c0 + lane) * 16) = v;
  }
}

template <int CH>
__device__ __forceinline__ void store_conv_state(const FusedArgs& p,
                                                 const int tid, const int bw,
                                                 const int h, const int c_first,
                                                 const int row0, const int row1) {
  const int T = p.T;
  const int64_t W = p.W;
  // Masked conv state of this slice's channels: rows T-3..T-1 of x, each
  // zeroed if a document starts in a later position of the row; rows before
  // the sequence start are zero.
  {
    const int nb = row1 - row0;
    int t_id = tid;
    asm volatile("" : "+v"(t_id));
    for (int idx = t_id; idx < nb * (CH / 2); idx += kThreads) {
      const int b = row0 + idx / (CH / 2);
      const int c_in = c_first + 2 * (idx % (CH / 2));
      if (c_in >= bw) continue;
      const int64_t c = h * bw + c_in;
      uint16_t* cache = (uint16_t*)p.cache_out + (int64_t)b * 3 * W + c;
      bool later_start = false;
#pragma unroll
      for (int kk = 2; kk >= 0; --kk) {
        const int t = T - 3 + kk;
        uint32_t v = 0;
        if (t >= 0 && !later_start)
          v = *reinterpret_cast<const uint32_t*>(
              (const uint16_t*)p.x + ((int64_t)b * T + t) * W + c);
        *reinterpret_cast<uint32_t*>(cache + (int64_t)kk * W) = v;
        if (t >= 0 && is_doc_start(p.segpos, p.seg_kind, (int64_t)b * T + t))
          later_start = true;
      }
    }
  }
}

// KS: k-steps of 16 (a head of bw <= 16 KS channels, zeros beyond bw).
// PACKED: gate weights in operand order (launch_pack_gate_weights), else as
// the reference lays them out.  GELU: y leaves as y * gelu(gate_branch), the
// block's join (recurrentgemma/torch/modules.py:627-628, 644).
// MANY: rows of at most 16 tokens, as many whole ones to a tile as go into it; what is
// a row of the batch elsewhere is a tile here.  (A row to a tile leaves most of it empty:
// figures at prefill_many_serve.)
template <int KS, bool PACKED, bool GELU, bool MANY>
__global__ void __launch_bounds__(kThreads)
block_prefill_slices_bf16_kernel(FusedArgs p, RowsOfTile many, int slices, int groups) {
  static_assert(PACKED || !MANY, "");
  using L = Layout<KS>;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  lds_byte* const lds3 = (lds_byte*)lds_raw;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bw = p.W / p.H;
  // Workgroups go to the eight XCDs in turn: the slices of a (row range, head)
  // pair, which read the same rows and one head's weights, are dealt to one
  // XCD (the grid is rounded up to whole rounds, the surplus exits).
  const int xcd = blockIdx.x & 7, in_xcd = blockIdx.x >> 3;
  const int pair = (in_xcd / slices) * 8 + xcd;
  if (pair >= groups * p.H) return;
  const int slice = in_xcd % slices;
  const int h = pair / groups;
  const int group = pair - h * groups;
  const int rows = MANY ? (p.B + many.rows - 1) / many.rows : p.B;
  const int row0 = (int)((int64_t)group * rows / groups);
  const int row1 = (int)((int64_t)(group + 1) * rows / groups);
  const int row_tokens = MANY ? many.rows * p.T : p.T;
  const int tiles_per_row = MANY ? 1 : (row_tokens + kTile - 1) / kTile;
  const int ntiles = (row1 - row0) * tiles_per_row;
  const int npasses = (ntiles + kTiles - 1) / kTiles;
  auto tokens_of = [&](int row) {  // (the last tile of MANY may hold fewer rows)
    return MANY && row + 1 == rows ? (p.B - row * many.rows) * p.T : row_tokens;
  };

  const uint32_t row_bytes = 2u * (uint32_t)p.W;
  const bool seg_is64 = p.seg_kind == kSegI64;
  const uint32_t seg_esize = seg_is64 ? 8u : 4u;

  // matrix role: tile `tt` of the pass, channels n0 .. n0 + 31 of the head
  const int tt = wave >> 1;
  const int half = wave & 1;
  const int n0 = slice * kSlice + half * 32;
  // conv role: the same tile, two channels of half of the head per lane
  const int conv_pair = half * 64 + lane;
  const bool conv_lane = conv_pair * 2 < KS * 16;
  const uint32_t conv_off = conv_pair * 2 < bw
                                ? 2u * (uint32_t)(h * bw + conv_pair * 2)
                                : kBufferOutOfRange;

  // Rows t0 - 3 .. t0 + 31 of this wave's tile in pass i, and the positions of
  // rows t0 - 32 .. t0 + 31, one per lane.
  uint32_t raw[kConvRows + 3];
  uint32_t seg_lo = 1, seg_hi = 0;
  bool seg_in = false;
  // Which row and which of its tiles this wave's tile of a pass is; a step is
  // one pass.
  struct At {
    int row, k;  // row past the range: no tile
  };
  const int step_rows = kTiles / tiles_per_row, step_k = kTiles % tiles_per_row;
  auto step = [&](At& at) RG_INLINE {
    at.row += step_rows;
    at.k += step_k;
    if (at.k >= tiles_per_row) {
      at.k -= tiles_per_row;
      ++at.row;
    }
  };
  At now = {row0 + tt / tiles_per_row, tt % tiles_per_row};
  At asked = now;
  auto request = [&]() RG_INLINE {  // ... of the pass `asked` stands at
    const bool any = asked.row < row1;
    const int b = any ? asked.row : row0;
    const int t0 = asked.k * kTile;
    step(asked);
    const int T = tokens_of(b);
    const uint32_t seq_bytes = (uint32_t)T * row_bytes;  // < 2^31 (launcher)
    const char* base = (const char*)p.x + (int64_t)b * row_tokens * row_bytes;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(base, any ? seq_bytes : 0);
    const __amdgpu_buffer_rsrc_t rhalo = make_rsrc(base, any && t0 ? seq_bytes : 0);
    // (the whole offset in the vector part, which the descriptor checks: rows
    // past the end of the sequence read as zeros, and so do the three before
    // its start, through a descriptor of no bytes)
    const uint32_t off = conv_off + (uint32_t)t0 * row_bytes;
#pragma unroll
    for (int r = 0; r < kConvRows + 3; ++r)
      raw[r] = __builtin_amdgcn_raw_buffer_load_b32(
          r < 3 ? rhalo : rx,
          r < 3 && t0 == 0 ? off : off + (uint32_t)(r - 3) * row_bytes, 0, 0);
    const int t = t0 + lane - 32;
    seg_in = any && t >= 0 && t < T;
    const char* seg_row =
        (const char*)p.segpos + (int64_t)b * row_tokens * seg_esize;  // (uniform)
    const uint32_t at = (uint32_t)(seg_in ? t : 0) * seg_esize;
    seg_lo = *reinterpret_cast<const uint32_t*>(seg_row + at);
    seg_hi = seg_is64 ? *reinterpret_cast<const uint32_t*>(seg_row + at + 4) : 0u;
  };
  // Document starts: bit j is row t0 - 32 + j
  auto starts_mask = [&]() RG_INLINE -> uint64_t {
    return __ballot(seg_in && (seg_lo | seg_hi) == 0u);
  };

  // Where the conv is cut: bit j, row j - 3 of the tile
  auto cuts_of = [&](uint64_t mask) RG_INLINE -> uint64_t {
    return mask >> 29 | (MANY ? (uint64_t)many.opens << 3 : 0);
  };

  // (MANY: beside the first rows its registers do not suffice for the weights)
  if (!PACKED || MANY) load_weights<KS, PACKED>(p, lane, bw, h, n0);
  request();
  if (PACKED && !MANY) load_weights<KS, true>(p, lane, bw, h, n0);
  fill_taps<L>(p, lds_raw, tid, bw, h);
  if (tt == 0) fill_gate_values<L>(p, lds_raw, lane, bw, h, n0, half * 32);
  __syncthreads();  // taps, per-channel values

  // ---- conv -----------------------------------------------------------------
  struct Conv {
    uint32_t w10[2], w32[2];
    float bias[2];
    uint32_t p1[2], p2[2];  // time pairs of the two rows before the next
  };
  auto conv_begin = [&](Conv& c) RG_INLINE {
    const u32x4 t0 =
        *reinterpret_cast<lds_u32x4*>(lds3 + L::taps + conv_pair * 32);
    const f32x2 t1 =
        *reinterpret_cast<lds_f32x2*>(lds3 + L::taps + conv_pair * 32 + 16);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      c.w10[e] = t0[e];
      c.w32[e] = t0[2 + e];
      c.bias[e] = t1[e];
    }
    pair_up(raw[0], raw[1], c.p2[0], c.p2[1]);
    pair_up(raw[1], raw[2], c.p1[0], c.p1[1]);
  };
  const uint32_t conv_out = (uint32_t)(tt * kTile) * L::row + conv_pair * 4;
  auto conv_store = [&](int buf, int r, const float (&o)[2]) {
    if (conv_lane)
      *reinterpret_cast<lds_u32*>(lds3 + buf * L::buffer + conv_out +
                                  r * L::row) = pack_bf16x2(o[0], o[1]);
  };
  // rows 2 j and 2 j + 1 of the tile
  auto conv_rows = [&](Conv& c, int buf, int j) RG_INLINE {
    uint32_t e[2], o[2];
    pair_up(raw[2 * j + 3], raw[2 * j + 4], e[0], e[1]);
#pragma unroll
    for (int i = 0; i < 2; ++i) o[i] = __builtin_amdgcn_alignbit(e[i], c.p1[i], 16);
    float even[2], odd[2];
    conv4_dot_row_pair(c.p2, o, c.p1, e, c.w10, c.w32, c.bias, even, odd);
    conv_store(buf, 2 * j, even);
    conv_store(buf, 2 * j + 1, odd);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      c.p1[i] = e[i];
      c.p2[i] = o[i];
    }
  };
  // the same rows with the history cut where a document starts (bit j of
  // `cuts`: row j - 3 of the tile), same products in the same order
  auto conv_with_cuts = [&](int buf, uint64_t cuts) RG_INLINE {
    Conv c;
    conv_begin(c);
    uint32_t before = 0;
    c.p1[0] = c.p1[1] = c.p2[0] = c.p2[1] = 0;
#pragma unroll
    for (int j = 0; j < kConvRows + 3; ++j) {
      if ((cuts >> j) & 1u) {
        before = 0;
        c.p1[0] = c.p1[1] = c.p2[0] = c.p2[1] = 0;
      }
      uint32_t pt[2];
      pair_up(before, raw[j], pt[0], pt[1]);
      if (j >= 3) {
        float o[2];
        conv4_dot_x2(c.p2, pt, c.w10, c.w32, c.bias, o);
        conv_store(buf, j - 3, o);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        c.p2[e] = c.p1[e];
        c.p1[e] = pt[e];
      }
      before = raw[j];
    }
  };

  // ---- pass 0's conv, pass 1's rows ----------------------------------------
  uint64_t mask = starts_mask();
  auto convolve = [&](int buf, uint64_t cuts) RG_INLINE {
    if (cuts != 0) {
      conv_with_cuts(buf, cuts);
    } else {
      Conv c;
      conv_begin(c);
#pragma unroll
      for (int j = 0; j < kConvRows / 2; ++j) conv_rows(c, buf, j);
    }
  };
  convolve(0, cuts_of(mask));
  uint32_t starts = (uint32_t)(mask >> 32);
  if (PACKED && !MANY && npasses > 1) request();
  lds_barrier();

  const uint32_t a_lane =
      (uint32_t)(tt * kTile + (lane & 31)) * L::row + 16u * (lane >> 5);
  // state behind the last tile of the pass before, of the row it belongs to
  float carry = 0.0f;
  int until = 0;

  // (the last pass apart: it has no conv to do, and accumulators that two
  // paths lead to would be copied behind their matrix instructions)
  auto pass = [&](int i, auto MORE) RG_INLINE {
    constexpr bool more = decltype(MORE)::value;
    const int buf = i & 1;
    const bool any = now.row < row1;
    const bool active = any && n0 < bw;
    const int b = any ? now.row : row0;
    const int k_in_row = now.k;
    const int t0 = k_in_row * kTile;
    step(now);
    // the next pass's conv between the matrix instructions, then the rows of
    // the one after
    // (weights in the reference layout, and MANY, which has one pass or two: the conv
    // runs before the matrix instructions -- between them registers do not suffice)
    if ((!PACKED || MANY) && more) {
      request();
      mask = starts_mask();
      convolve(buf ^ 1, cuts_of(mask));
    }
    f32x16 acc_x, acc_a;
    if constexpr (PACKED && !MANY && more) {
      mask = starts_mask();
      const uint64_t cuts = cuts_of(mask);
      Conv c;
      conv_begin(c);
      matrix_tile<KS>(lds3, a_lane + buf * L::buffer, acc_x, acc_a, [&](auto KSTEP) RG_INLINE {
        constexpr int ks = decltype(KSTEP)::value;
        // (the pairs j of rows with floor(j KS / pairs) == ks)
        constexpr int pairs = kConvRows / 2;
        constexpr int first = (ks * pairs + KS - 1) / KS;
        constexpr int last = ((ks + 1) * pairs + KS - 1) / KS;
        static_for<first, last>([&](auto J) RG_INLINE { conv_rows(c, buf ^ 1, decltype(J)::value); });
      });
      if (__builtin_expect(cuts != 0, 0)) conv_with_cuts(buf ^ 1, cuts);
      if (i + 2 < npasses) request();
    } else {
      matrix_tile<KS>(lds3, a_lane + buf * L::buffer, acc_x, acc_a, [](auto) RG_INLINE {});
    }
    gate_and_scan<L, GELU, MANY>(
        p, many, lds3, lane, wave, bw, h, n0, half * 32, tt, buf, tiles_per_row,
        TileAt{b, t0, k_in_row, any, active, starts, tokens_of(b)}, acc_x, acc_a,
        carry, until);
    starts = (uint32_t)(mask >> 32);
  };
  for (int i = 0; i + 1 < npasses; ++i) pass(i, std::true_type{});
  pass(npasses - 1, std::false_type{});

  if (p.cache_out)
    store_conv_state<kSlice>(p, tid, bw, h, slice * kSlice,
                             MANY ? row0 * many.rows : row0,
                             MANY ? min(row1 * many.rows, p.B) : row1);
}

// Heads of at most 176 channels (the paper presets): two slices of 96, and the
// waves of a workgroup specialised.  Six of them multiply, two teams of three groups
// of 32 channels that take the row's tiles of 32 tokens in turn, one phase apart: while
// one team has its matrix instructions (phase M) the other, on the same SIMDs, has its
// gates and the recurrence (phase G), as in rg_prefill_teams.hip.  Two do nothing but
// the conv of the tiles to come, beside the multiplying waves that have a SIMD to
// themselves otherwise: 32 heads x 2 slices x 4 rows are exactly one workgroup per CU
// where slices of 64 are one and a half.
//
// Phase p: M of tile p, G of tile p - 1; conv of tile p + 2's first 128 channels and of
// tile p + 1's others.  A workgroup barrier behind every phase; the state goes from
// tile to tile through LDS, and so the tokens are walked in their order.
//
// What bounds it: vector issue on the two SIMDs with two multiplying waves, which is
// busy all of the time with the join (840 slots a phase, 22 matrix instructions among
// them, of 1.6 us) and three quarters of it without (1.25 us); the other two have a
// tenth less.  us, all four multiplying and both converting waves of a tile pair in the
// same phases, the state by (prod a, state from zero) as in the form above / now, W5632
// H32: B4 T2048 115 / 88, joined 126 / 109; B16 T2048 433 / 329, joined 476 / 414; B40
// T300 183 / 144, joined 201 / 173; B64 T33 75 / 66, joined 82 / 73; B16 T100 38 / 34,
// joined 42 / 38.
constexpr int kNarrowKS = 11, kNarrowTeams = 2, kNarrowGroups = 3;
constexpr int kNarrowSlice = 32 * kNarrowGroups;
constexpr int kNarrowPairs = kNarrowKS * 8;  // channel pairs of a head
constexpr int kNarrowRing = 4;  // conv tiles: two being made, one in M, one done with
constexpr int kNarrowRaw = 6;   // tiles of raw rows: four on their way, two being read
struct NarrowLayout {
  static constexpr int row = (kNarrowKS * 16 + 8) * 2;
  static constexpr int tile = kTile * row;
  static constexpr int patch = kNarrowRing * tile;
  // (a wave's output patch: 16 tokens x 32 channels; the upper lanes' eight rows
  // another 64 bytes on, in other banks)
  static constexpr int patch_upper = 8 * kPatchStride + 64;
  static constexpr int patch_wave = patch_upper + 8 * kPatchStride;
  // raw rows, 35 of a tile
  static constexpr int raw_pieces = kNarrowKS * 2, raw_row = 16 * raw_pieces;
  static constexpr int raw_loads = ((kTile + 3) * raw_pieces + 63) / 64;
  static constexpr int raw_tile = raw_loads * 1024;
  static constexpr int raw = patch + kNarrowTeams * kNarrowGroups * patch_wave;
  static constexpr int state = raw + kNarrowRaw * raw_tile;
  static constexpr int taps = state + kNarrowSlice * 4;
  static constexpr int gates = taps + 128 * 32;
  static constexpr int total = gates + kNarrowSlice * 16;
  static_assert(taps % 16 == 0 && total <= 160 * 1024, "LDS of one CU");
};

// 16 bytes a lane from memory into LDS, 1 KB in a row.
__device__ __forceinline__ void load_to_lds(const __amdgpu_buffer_rsrc_t from,
                                            lds_byte* const to, const uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, to, 16, off, 0, 0, 0);
}

// A bf16 value of LDS into the high half of a zeroed register: as a float without a
// shift.  (The wait for it is the reader's.)
template <int OFFSET>
__device__ __forceinline__ uint32_t read_bf16_high(uint32_t at) {
  uint32_t v;
  asm volatile("v_mov_b32 %0, 0\n\tds_read_u16_d16_hi %0, %1 offset:%2"
               : "=&v"(v)
               : "v"(at), "n"(OFFSET));
  return v;
}

template <bool PACKED, bool GELU>
__global__ void __launch_bounds__(kThreads)
block_prefill_narrow_bf16_kernel(FusedArgs p, int slices, int groups) {
  using L = NarrowLayout;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  lds_byte* const lds3 = (lds_byte*)lds_raw;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bw = p.W / p.H;
  const int xcd = blockIdx.x & 7, in_xcd = blockIdx.x >> 3;
  const int pair = (in_xcd / slices) * 8 + xcd;
  if (pair >= groups * p.H) return;
  const int slice = in_xcd % slices;
  const int h = pair / groups;
  const int group = pair - h * groups;
  const int row0 = (int)((int64_t)group * p.B / groups);
  const int row1 = (int)((int64_t)(group + 1) * p.B / groups);
  const int T = p.T;
  const int64_t W = p.W;
  const int tiles_per_row = (T + kTile - 1) / kTile;
  const int ntiles = (row1 - row0) * tiles_per_row;
  const uint32_t row_bytes = 2u * (uint32_t)p.W;
  const uint32_t seq_bytes = (uint32_t)T * row_bytes;  // < 2^31 (launcher)
  const bool seg_is64 = p.seg_kind == kSegI64;
  const uint32_t seg_esize = seg_is64 ? 8u : 4u;

  const bool convolves = wave >= kNarrowTeams * kNarrowGroups;
  // this wave's tiles: every second, from this one on
  const int first = convolves ? wave - kNarrowTeams * kNarrowGroups
                              : wave / kNarrowGroups;
  struct At {  // a tile: row (past the range: none), and which of the row's
    int row, k;
  };
  const int step_rows = kNarrowTeams / tiles_per_row;
  const int step_k = kNarrowTeams % tiles_per_row;
  auto step = [&](At& at) RG_INLINE {
    at.row += step_rows;
    at.k += step_k;
    if (at.k >= tiles_per_row) {
      at.k -= tiles_per_row;
      ++at.row;
    }
  };
  const At begin = {row0 + first / tiles_per_row, first % tiles_per_row};
  // positions of rows t0 - 32 .. t0 + 31 of the tile a wave asks for
  uint32_t seg_lo = 1, seg_hi = 0;
  bool seg_in = false;
  // (no branch: a load on one of two paths is waited for, with all before it, on both)
  auto request_positions = [&](const At& at) RG_INLINE {
    const bool any = at.row < row1;
    const uint32_t bytes = (uint32_t)T * seg_esize;
    const __amdgpu_buffer_rsrc_t rseg = make_rsrc(
        (const char*)p.segpos + (int64_t)(any ? at.row : row0) * bytes, any ? bytes : 0u);
    const int t = at.k * kTile + lane - 32;
    seg_in = any && (uint32_t)t < (uint32_t)T;
    const uint32_t off = seg_in ? (uint32_t)t * seg_esize : kBufferOutOfRange;
    seg_lo = __builtin_amdgcn_raw_buffer_load_b32(rseg, off, 0, 0);
    seg_hi = __builtin_amdgcn_raw_buffer_load_b32(
        rseg, seg_is64 ? off + 4u : kBufferOutOfRange, 0, 0);
  };
  auto starts_mask = [&]() RG_INLINE -> uint64_t {
    return __ballot(seg_in && (seg_lo | seg_hi) == 0u);
  };
  // Where a token's conv output lies in its tile: a lane of the matrix result has
  // rows 0-3, 8-11, .. (upper lanes 4-7, 12-15, ..), and gets sixteen tokens in a row.
  auto conv_row = [](int t) RG_INLINE {
    return 8 * ((t & 15) >> 2) + (t & 3) + 4 * (t >> 4);
  };
  auto conv_at = [](int tile) RG_INLINE {
    return (uint32_t)((tile % kNarrowRing) * L::tile);
  };
  fill_taps<L>(p, lds_raw, tid, bw, h);
  // Behind every phase.  (lds_barrier would wait for the raw rows on their way into
  // LDS, too: whoever reads them waits for them, two phases on.)
  auto phase_barrier = []() RG_INLINE {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto wait_loads = []() RG_INLINE {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L::raw_loads) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  if (convolves) {
    // ---- conv: channel pairs 0-63 of the head, 32 rows a lane; then the 24
    //      others, 16 rows a lane (the upper lanes the later ones) -------------
    const int pair_b = 64 + (lane & 31);
    const bool lane_b = pair_b < kNarrowPairs;
    const int row_b = (lane >> 5) * 16;
    constexpr int kRowsB = 16;
    // Raw rows t0 - 3 .. t0 + 31 of a tile as the memory pipe writes them into LDS,
    // 22 pieces of 16 bytes each (zeros beyond the head and the sequence), two tiles
    // of each of the two waves.  (As 54 loads of four bytes a lane into registers, two
    // rows a load at best, the conv took longer than the other waves' phases: B4 T2048
    // W5632 110 us, joined 124.)
    uint32_t piece[L::raw_loads];
#pragma unroll
    for (int j = 0; j < L::raw_loads; ++j) {
      const int q = 64 * j + lane, r = q / L::raw_pieces, c = q % L::raw_pieces;
      piece[j] = r < kTile + 3 && 8 * c < bw
                     ? (uint32_t)((r - 3) * (int)row_bytes) +
                           2u * (uint32_t)(h * bw) + 16u * c
                     : kBufferOutOfRange;
    }
    At asked = begin, asked_positions = begin;
    auto raw_at = [](int tile) RG_INLINE {
      return (uint32_t)(L::raw + (tile % kNarrowRaw) * L::raw_tile);
    };
    auto request = [&](int tile) RG_INLINE {  // (the one that `asked` stands at)
      const bool any = asked.row < row1;
      const uint32_t before = (uint32_t)(asked.k * kTile) * row_bytes;
      const __amdgpu_buffer_rsrc_t rx = make_rsrc(
          (const char*)p.x + (int64_t)(any ? asked.row : row0) * seq_bytes,
          any ? seq_bytes : 0);
#pragma unroll
      for (int j = 0; j < L::raw_loads; ++j)
        load_to_lds(rx, lds3 + raw_at(tile) + 1024 * j, piece[j] + before);
      step(asked);
    };
    // ROWS rows from raw rows; bit j of `cuts`: raw row j starts a document
    auto convolve = [&](const uint32_t raw_from, auto ROWS, const int pair_of_lane,
                        const uint32_t out, const bool store,
                        const uint64_t cuts) RG_INLINE {
      constexpr int rows = decltype(ROWS)::value;
      uint32_t raw[rows + 3];
#pragma unroll
      for (int r = 0; r < rows + 3; ++r)
        raw[r] = *reinterpret_cast<lds_u32*>(lds3 + raw_from + r * L::raw_row);
      uint32_t w10[2], w32[2];
      float bias[2];
      const u32x4 t0 =
          *reinterpret_cast<lds_u32x4*>(lds3 + L::taps + pair_of_lane * 32);
      const f32x2 t1 = *reinterpret_cast<lds_f32x2*>(lds3 + L::taps +
                                                     pair_of_lane * 32 + 16);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        w10[e] = t0[e];
        w32[e] = t0[2 + e];
        bias[e] = t1[e];
      }
      auto put = [&](int r, const float (&o)[2]) RG_INLINE {
        if (store)
          *reinterpret_cast<lds_u32*>(lds3 + out + conv_row(r) * L::row) =
              pack_bf16x2(o[0], o[1]);
      };
      uint32_t p1[2], p2[2];
      if (__builtin_expect(__any(cuts != 0), 0)) {
        uint32_t before = 0;
        p1[0] = p1[1] = p2[0] = p2[1] = 0;
#pragma unroll
        for (int j = 0; j < rows + 3; ++j) {
          const bool cut = (cuts >> j) & 1u;
          uint32_t pt[2];
          pair_up(cut ? 0u : before, raw[j], pt[0], pt[1]);
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            p1[e] = cut ? 0u : p1[e];
            p2[e] = cut ? 0u : p2[e];
          }
          if (j >= 3) {
            float o[2];
            conv4_dot_x2(p2, pt, w10, w32, bias, o);
            put(j - 3, o);
          }
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            p2[e] = p1[e];
            p1[e] = pt[e];
          }
          before = raw[j];
        }
        return;
      }
      pair_up(raw[0], raw[1], p2[0], p2[1]);
      pair_up(raw[1], raw[2], p1[0], p1[1]);
#pragma unroll
      for (int j = 0; j < rows / 2; ++j) {
        uint32_t e[2], o[2];
        pair_up(raw[2 * j + 3], raw[2 * j + 4], e[0], e[1]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          o[i] = __builtin_amdgcn_alignbit(e[i], p1[i], 16);
        float even[2], odd[2];
        conv4_dot_row_pair(p2, o, p1, e, w10, w32, bias, even, odd);
        put(2 * j, even);
        put(2 * j + 1, odd);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          p1[i] = e[i];
          p2[i] = o[i];
        }
      }
    };
    uint64_t mask = 0;  // of the tile whose first part was made last
    auto make_a = [&](int tile) RG_INLINE {
      // the tile's raw rows, asked for three phases ago, and its positions (the rows of
      // the next tile of this wave may still be on their way)
      wait_loads();
      mask = starts_mask();
      request_positions(asked_positions);
      step(asked_positions);
      convolve(raw_at(tile) + lane * 4, std::integral_constant<int, kTile>{}, lane,
               conv_at(tile) + lane * 4, true, mask >> 29);
    };
    // (the wave that shares the SIMD has its phase G then: the loads, which hold a wave
    // 50 to 100 cycles each, where there is less of the conv)
    auto make_b = [&](int tile) RG_INLINE {
      request(tile + 2 * kNarrowTeams);
      convolve(raw_at(tile) + row_b * L::raw_row + pair_b * 4,
               std::integral_constant<int, kRowsB>{}, lane_b ? pair_b : 64,
               conv_at(tile) + 4 * (lane >> 5) * L::row + pair_b * 4, lane_b,
               (mask >> (29 + row_b)) & ((1u << (kRowsB + 3)) - 1u));
    };
    request(first);
    request_positions(asked_positions);
    step(asked_positions);
    request(first + kNarrowTeams);
    __syncthreads();  // taps
    make_a(first);
    if (first == 0) make_b(0);
    phase_barrier();
    int phase = 0, tile = 2;
    if (first == 1) {
      make_b(1);
      phase_barrier();
      phase = 1;
      tile = 3;
    }
    for (; phase < ntiles; phase += 2, tile += 2) {
      if (tile < ntiles) make_a(tile);
      phase_barrier();
      if (tile < ntiles) make_b(tile);
      if (phase + 1 < ntiles) phase_barrier();
    }
  } else {
    const int team = first;
    const int c0 = 32 * (wave % kNarrowGroups);
    const int n0 = slice * kNarrowSlice + c0;
    load_weights<kNarrowKS, PACKED>(p, lane, bw, h, n0);
    if (team == 0) fill_gate_values<L>(p, lds_raw, lane, bw, h, n0, c0);
    __syncthreads();  // taps
    phase_barrier();  // the first conv tiles, the gate values
    const f32x4 per_channel = *reinterpret_cast<lds_f32x4*>(
        lds3 + L::gates + (c0 + (lane & 31)) * 16);
    const float bias_x = per_channel[0], bias_a = per_channel[1];
    const float inv_decay = per_channel[2];
    const uint32_t a_lane = (uint32_t)(lane & 31) * L::row + 16u * (lane >> 5);
    const uint32_t xc_lane = 4u * (lane >> 5) * L::row + 2u * (uint32_t)(n0 + (lane & 31));
    const uint32_t patch_at = L::patch + wave * L::patch_wave + (lane >> 5) * L::patch_upper;
    const uint32_t patch_w = patch_at + 2u * (lane & 31);
    const uint32_t patch_r =
        patch_at + (uint32_t)((lane >> 2) & 7) * kPatchStride + 16u * (lane & 3);
    const bool ch_valid = n0 + (lane & 31) < bw;
    // (8 channels a lane: all of them channels of the head or none)
    const uint32_t y_lane =
        n0 + 8 * (lane & 3) < bw
            ? (uint32_t)(16 * (lane >> 5) + ((lane >> 2) & 7)) * row_bytes +
                  2u * (uint32_t)(h * bw + n0) + 16u * (lane & 3)
            : kBufferOutOfRange;
    const uint32_t state_at = L::state + 4u * (uint32_t)(c0 + (lane & 31));
    const uint32_t ch_bytes = ch_valid ? 4u * (uint32_t)(h * bw + n0 + (lane & 31))
                                       : kBufferOutOfRange;
    auto state_row = [&](const float* base, int b, bool any) RG_INLINE {
      return make_rsrc(base + (int64_t)b * W, base && any ? 4u * (uint32_t)p.W : 0u);
    };
    float h0 = 0.0f;  // of a tile that opens its row

    f32x16 acc_x, acc_a;
    uint32_t xr[16];  // conv outputs, this lane's tokens, as floats
    u32x4 y_pending[2];
    int y_row = -1;  // where they belong: row (none yet) and first token
    uint32_t y_at = 0;
    At at = begin;

    auto rows_of = [&](const void* base, int b, bool any) RG_INLINE {
      return make_rsrc((const char*)base + (int64_t)b * seq_bytes, any ? seq_bytes : 0u);
    };
    // (a lane past the head's channels keeps its offset out of every descriptor)
    auto y_offset = [&](uint32_t before) RG_INLINE {
      return y_lane == kBufferOutOfRange ? kBufferOutOfRange : y_lane + before;
    };
    auto store_pending = [&]() RG_INLINE {
      const __amdgpu_buffer_rsrc_t ry = rows_of(p.y, y_row < 0 ? row0 : y_row, y_row >= 0);
      buffer_store_16(y_pending[0], ry, y_offset(y_at), 0);
      buffer_store_16(y_pending[1], ry, y_offset(y_at + 8u * row_bytes), 0);
    };
    y_pending[0] = y_pending[1] = u32x4{0, 0, 0, 0};
    u32x4 gate_rows[2];  // the gate branch's values, then gelu of them

    // What phase G reads of tile `at`, asked for a tile of this team ahead and in front
    // of the outputs of the tile before (loads and stores are waited for in order).
    auto request = [&]() RG_INLINE {
      const bool any = at.row < row1;
      request_positions(at);
      h0 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          state_row(p.h0, any ? at.row : row0, any && at.k == 0), ch_bytes, 0, 0));
      if (GELU) {
        const __amdgpu_buffer_rsrc_t rgate =
            rows_of(p.gate_branch, any ? at.row : row0, any);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          gate_rows[j] = __builtin_amdgcn_raw_buffer_load_b128(
              rgate, y_offset((uint32_t)(at.k * kTile + 8 * j) * row_bytes), 0, 0);
      }
    };

    // ---- phase M: the tile's matrix instructions; y of this team's tile before ----
    auto phase_m = [&](int tile) RG_INLINE {
      const uint32_t tile_at = conv_at(tile);
      store_pending();
      const uint32_t x_at = tile_at + xc_lane;
      __builtin_amdgcn_s_setprio(1);
      matrix_tile<kNarrowKS>(lds3, tile_at + a_lane, acc_x, acc_a, [&](auto KSTEP) RG_INLINE {
        constexpr int ks = decltype(KSTEP)::value;
        // the conv outputs for the gate arithmetic (in phase G)
        if constexpr (ks >= kNarrowKS - 4) {
          static_for<4 * (ks - kNarrowKS + 4), 4 * (ks - kNarrowKS + 5)>([&](auto I) RG_INLINE {
            constexpr int i = decltype(I)::value;
            xr[i] = read_bf16_high<(8 * (i >> 2) + (i & 3)) * L::row>(x_at);
          });
        }
      });
      __builtin_amdgcn_s_setprio(0);
      // gelu here, the gates in phase G.  (us, B4 T2048 W5632: joined 112.1, with gelu in
      // phase G 115.4; plain 90.4, with 4, 8 or 16 of the lane's input gates here 91.1,
      // 92.3, 98.4)
      if (GELU) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int k = 0; k < 4; ++k) gate_rows[j][k] = gelu_bf16x2(gate_rows[j][k]);
        asm volatile("" : "+v"(gate_rows[0]), "+v"(gate_rows[1]));
      }
    };
    // ---- phase G: gates, recurrence, outputs ---------------------------------------
    auto phase_g = [&](auto GENERAL, uint32_t tile_starts) RG_INLINE {
      constexpr bool general = decltype(GENERAL)::value;
      const int t0 = at.k * kTile;
      // the state before the tile
      float before = *reinterpret_cast<__attribute__((address_space(3))) float*>(
          lds3 + state_at);
      before = at.k == 0 ? h0 : before;
      float xn[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float gx = __builtin_amdgcn_rcpf(
            1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(acc_x[i], -kLog2e, bias_x)));
        acc_a[i] = __builtin_amdgcn_exp2f(gate_exponent(
            __builtin_amdgcn_exp2f(__builtin_fmaf(acc_a[i], -kLog2e, bias_a)),
            inv_decay));
        xn[i] = __uint_as_float(xr[i]) * gx;
      }
      if (general) {
        // document start: a = 0; past the end of the row: identity
        int token0 = (lane >> 5) * 16;
        asm volatile("" : "+v"(token0));
        const uint32_t mine = tile_starts >> token0;
        const int left = T - t0 - token0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          acc_a[i] = (mine >> i) & 1u ? 0.0f : acc_a[i];
          acc_a[i] = i < left ? acc_a[i] : 1.0f;
          xn[i] = i < left ? xn[i] : 0.0f;
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i)
        xn[i] *= __builtin_amdgcn_sqrtf(__builtin_fmaf(-acc_a[i], acc_a[i], 1.0f));
      // walked twice: right for the lower lanes, whose end goes to the upper ones,
      // then from each half's own incoming state
      float e1 = before;
#pragma unroll
      for (int i = 0; i < 16; ++i) e1 = __builtin_fmaf(acc_a[i], e1, xn[i]);
      const auto sw = __builtin_amdgcn_permlane32_swap(
          __float_as_uint(before), __float_as_uint(e1), false, false);
      float hh = __uint_as_float(sw[0]);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float hv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          hh = __builtin_fmaf(acc_a[4 * g + q], hh, xn[4 * g + q]);
          hv[q] = hh;
        }
        const uint32_t y01 = pack_bf16x2(hv[0], hv[1]);
        const uint32_t y23 = pack_bf16x2(hv[2], hv[3]);
        asm volatile(
            "ds_write_b16 %0, %1 offset:%3\n\t"
            "ds_write_b16_d16_hi %0, %1 offset:%4\n\t"
            "ds_write_b16 %0, %2 offset:%5\n\t"
            "ds_write_b16_d16_hi %0, %2 offset:%6"
            :
            : "v"(patch_w), "v"(y01), "v"(y23), "n"((4 * (g & 1)) * kPatchStride),
              "n"((4 * (g & 1) + 1) * kPatchStride),
              "n"((4 * (g & 1) + 2) * kPatchStride),
              "n"((4 * (g & 1) + 3) * kPatchStride)
            : "memory");
        if (g & 1) {
          // (the LDS unit executes a wave's instructions in order)
          y_pending[g >> 1] = *reinterpret_cast<lds_u32x4*>(lds3 + patch_r);
          asm volatile("" ::: "memory");
        }
      }
      // the state behind the tile: the upper lanes' end
      if (lane >= 32) {
        *reinterpret_cast<__attribute__((address_space(3))) float*>(lds3 + state_at) = hh;
        if (at.k == tiles_per_row - 1)
          __builtin_amdgcn_raw_buffer_store_b32(
              __float_as_uint(hh), state_row(p.h_last, at.row, true), ch_bytes, 0, 0);
      }
      if (GELU) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int k = 0; k < 4; ++k)
            y_pending[j][k] = mul_bf16x2(y_pending[j][k], gate_rows[j][k]);
      }
      // (done here: behind the loads of the next tile they would be waited for)
      asm volatile("" : "+v"(y_pending[0]), "+v"(y_pending[1]));
      __builtin_amdgcn_sched_barrier(0);
      y_row = at.row;
      y_at = (uint32_t)t0 * row_bytes;
    };

    request();
    if (team == 1) phase_barrier();
    for (int tile = team; tile < ntiles; tile += kNarrowTeams) {
      phase_m(tile);
      phase_barrier();
      const uint32_t starts = (uint32_t)(starts_mask() >> 32);
      if (__builtin_expect(starts != 0 || (at.k + 1) * kTile > T, 0))
        phase_g(std::true_type{}, starts);
      else
        phase_g(std::false_type{}, starts);
      step(at);
      request();
      if (tile + 1 < ntiles) phase_barrier();
    }
    store_pending();
  }
  if (p.cache_out)
    store_conv_state<kNarrowSlice>(p, tid, bw, h, slice * kNarrowSlice, row0, row1);
}
// How many ranges the rows are cut into, and the time that takes: workgroups
// come in rounds of one per CU, and each costs a fixed part (weights, the
// first rows) and its passes.  (Pairs are launched in eights: 85 with three slices each are
// 264 workgroups, and the last eight a round of their own.)
struct Split {
  int groups;
  float us;
  int64_t rounds, passes;  // passes: of a workgroup
};
Split best_split(int B, int H, int T, int slices, int tiles, float fixed_us,
                 float pass_us) {
  const int64_t tiles_per_row = (T + kTile - 1) / kTile;
  Split best{1, 1e30f, 1, 1};
  for (int r = 1; r <= 9; ++r) {  // r workgroups per CU, and every row apart
    int64_t groups = r == 9 ? B : 256 * r / slices / 8 * 8 / H;
    if (groups < 1) groups = 1;
    if (groups > B) groups = B;
    const int64_t rows = (B + groups - 1) / groups;
    const int64_t passes = (rows * tiles_per_row + tiles - 1) / tiles;
    const int64_t rounds = ((groups * H + 7) / 8 * 8 * slices + 255) / 256;
    const float us = rounds * (fixed_us + passes * pass_us);
    if (us < best.us) best = Split{(int)groups, us, rounds, passes};
  }
  return best;
}

template <class K, class... Extra>
hipError_t launch_one(K kernel, OncePerDevice& once, int lds, const FusedArgs& a,
                      int slices, int groups, hipStream_t s, Extra... extra) {
  hipError_t e = set_max_dynamic_lds(once, (const void*)kernel, lds);
  if (e != hipSuccess) return e;
  const int64_t rounds = ((int64_t)groups * a.H + 7) / 8;
  if (rounds * 8 * slices > 0x7fffffff) return hipErrorInvalidValue;
  kernel<<<dim3((unsigned)(rounds * 8 * slices)), kThreads, lds, s>>>(
      a, extra..., slices, groups);
  return hipGetLastError();
}

// The form and the split of a shape.
enum Form { kSlices16, kSlices11, kNarrow };
struct Plan {
  Form form;
  int slices;
  Split split;
};
Plan plan(int B, int H, int T, int bw, bool joined) {
  // fixed part and pass of a workgroup, us (measured with every CU at work:
  // W2560 H10 T64 .. T448, W5632 H32 T16 .. T4096)
  const int slices = (bw + kSlice - 1) / kSlice;
  if (bw > kNarrowKS * 16)
    return Plan{kSlices16, slices,
                best_split(B, H, T, slices, kTiles, joined ? 5.8f : 6.2f,
                           joined ? 6.3f : 5.2f)};
  // Narrow heads: four tiles at once for few rows of up to 128 tokens, else the
  // specialised waves (whose walk in the tokens' order rounds states differently: the
  // form does not depend on the join, so that a joined call is a plain one and the join,
  // bit for bit).
  const Split wide = best_split(B, H, T, slices, kTiles, 6.2f, 5.2f);
  const int pairs = (bw + kNarrowSlice - 1) / kNarrowSlice;
  const Split roles = best_split(B, H, T, pairs, kNarrowTeams, 7.0f, 3.2f);
  // (two tiles a workgroup have the two teams one behind the other: while the four-tile
  // form's workgroups have a CU each that is ahead.  us, two teams / four tiles at once, 33
  // to 64 tokens, 1 to 32 pairs: 9.7 to 10.1 / 9.6 to 10.0, joined 10.4 to 10.8 / 10.0 to
  // 10.5; 64 pairs 10.1 to 10.2 / 10.0 to 10.5, joined 10.8 / 10.6; 85 pairs, in two rounds,
  // 10.0 / 18.0, 128 10.9 / 11.3, joined 11.8 / 12.1)
  const bool two_tiles = T > kTile && T <= 2 * kTile &&
                         ((int64_t)B * H + 7) / 8 * 8 * slices <= 256;
  if (two_tiles || wide.us <= roles.us) return Plan{kSlices11, slices, wide};
  return Plan{kNarrow, pairs, roles};
}

template <bool PACKED, bool GELU>
hipError_t launch_as(const FusedArgs& a, const Plan& p, hipStream_t s) {
  static OncePerDevice once[3];
  switch (p.form) {
    case kNarrow:
      return launch_one(block_prefill_narrow_bf16_kernel<PACKED, GELU>, once[0],
                        NarrowLayout::total, a,
                        p.slices, p.split.groups, s);
    case kSlices11:
      return launch_one(block_prefill_slices_bf16_kernel<11, PACKED, GELU, false>,
                        once[1], Layout<11>::total, a, p.slices,
                        p.split.groups, s, RowsOfTile{});
    default:
      return launch_one(block_prefill_slices_bf16_kernel<16, PACKED, GELU, false>,
                        once[2], Layout<16>::total, a, p.slices,
                        p.split.groups, s, RowsOfTile{});
  }
}

// Rows of at most 16 tokens, several to a tile.
constexpr int kManyTokens = kTile / 2;
Plan many_plan(int B, int H, int T, int bw) {
  const int rows = kTile / T, slices = (bw + kSlice - 1) / kSlice;
  return Plan{bw > kNarrowKS * 16 ? kSlices16 : kSlices11, slices,
              best_split((int)(((int64_t)B + rows - 1) / rows), H, kTile, slices, kTiles,
                         7.0f, 6.3f)};
}
template <bool GELU>
hipError_t launch_many(const FusedArgs& a, hipStream_t s) {
  const Plan p = many_plan(a.B, a.H, a.T, a.W / a.H);
  RowsOfTile many{kTile / a.T, 0u, 0u, 65536u / (uint32_t)a.T + 1u};
  for (int r = 0; r < many.rows; ++r) {
    many.opens |= 1u << (r * a.T);
    many.ends |= 1u << (r * a.T + a.T - 1);
  }
  static OncePerDevice once[2];
  if (p.form == kSlices11)
    return launch_one(block_prefill_slices_bf16_kernel<11, true, GELU, true>, once[0],
                      Layout<11>::total, a, p.slices, p.split.groups, s, many);
  return launch_one(block_prefill_slices_bf16_kernel<16, true, GELU, true>, once[1],
                    Layout<16>::total, a, p.slices, p.split.groups, s, many);
}

}  // namespace

// k-steps of 16 the packed weights of a head of bw channels are laid out for.
int gate_k_steps(int bw) { return bw <= kNarrowKS * 16 ? kNarrowKS : 16; }

// The whole-head form (rg_prefill_teams.hip): one workgroup per pair, 64 tokens in 4.35
// us (joined 6.65).
static float whole_heads_us(int B, int H, int T, bool joined) {
  const int64_t rounds = ((int64_t)B * H + 255) / 256;
  const int64_t tiles = (T + 63) / 64;
  return rounds * (joined ? 8.3f + 6.65f * tiles : 8.8f + 4.35f * tiles);
}

bool prefill_slices_serve(int B, int H, int T, bool joined) {
  const int64_t rounds = ((int64_t)B * H + 255) / 256;
  const float whole = whole_heads_us(B, H, T, joined);
  // (beyond two rounds of pairs four times as many workgroups read the rows
  // anew from memory, which the estimate does not know: B46 T48 W4096 39, here
  // 44)
  return plan(B, H, T, 256, joined).split.us < (rounds > 2 ? 0.75f : 1.0f) * whole;
}

// Rows of a few tokens, several to a tile, where that takes fewer passes than a row to a
// tile (its own pass is 0.5 to 1 us longer), or than whole heads by the workgroup.  us,
// joined, otherwise / so: W4096 B24 T1 18.7 / 12.3, T9 19.5 / 14.0, W5632 H32 B24 T3 27.1 /
// 13.0, T9 34.8 / 13.9, B64 T1 26.1 / 13.3, T9 50 / 31; with one pass either way W2560 B24
// T9 13.2 / 14.2, B2 T1 11.0 / 11.8.
//
// Beyond 512 pairs rg_recurrent_core's form is gate GEMM + scan.  256-wide heads stay
// there: its outputs are those of the two calls, bit for bit.  Narrower ones go by what
// either takes, fitted to 990 calls (heads of 136 to 248, 1 to 32 of them, 64 to 600 rows of
// 1 to 16 tokens): apart within 20 %, here within 15 % but for single passes (8.2 a pass,
// 9.3 with a state carried in).  us, here / apart: joined, 176 H10 B64 T16 12.8 / 28.3, B300
// 46 / 66, 136 H32 B600 T9 175 / 188; without a conv, which costs the two calls a third, 136
// H10 B300 T16 42.0 / 39.7, H32 B600 T9 166 / 124, 176 H1 B600 T3 11.9 / 16.
bool prefill_many_serve(int B, int H, int T, int bw, bool joined, bool conv, bool state) {
  if (B < 2 || T > kManyTokens || bw <= 128 || bw > 256 || bw % 8) return false;
  const Split split = many_plan(B, H, T, bw).split;
  const float here = split.us;
  if ((int64_t)B * H > 512) {
    const float rows = 1e-6f * (float)B * (float)(H * bw), elements = rows * (float)T;
    const float apart = (conv ? 17.2f + 7.5f * rows + 4.6f * elements
                              : 14.0f + 5.2f * rows + 3.6f * elements) +
                        (joined ? 1.8f + 0.95f * elements : 0.0f);
    return bw < 256 &&
           split.rounds * (5.0f + (state ? 9.3f : 8.4f) * split.passes) < apart;
  }
  const float apart = plan(B, H, T, bw, joined).split.us;
  return here < (bw < 256 || prefill_slices_serve(B, H, T, joined)
                     ? apart
                     : whole_heads_us(B, H, T, joined));
}

bool prefill_narrow_pays(int B, int H, int T, int W) {
  // Against the gate GEMM, the scan and the join as passes of their own: 34 us +
  // 0.0255 us a token of width 5632, as measured at 32 heads of 176.  Checked at 8,
  // 20 and 32 heads of 136, 152, 176, 184, 200 and 248 channels, one row of 64 to 64
  // rows of 128 and 16 of 2048, joined and not, from a graph (576 pairs of times):
  // whatever it sends here is faster here, by 6 % or more (us, apart / here, joined: 8
  // heads of 136 B8 T64 22 / 11, B16 T2048 197 / 112; 20 of 200 B32 T512 310 / 262; 32
  // of 176 B4 T2048 228 / 118, B64 T27 77 / 46; 32 of 248 B4 T4096 561 / 406, B64 T128
  // 305 / 223).  48 times it keeps rows of 1000 to 4096 tokens apart that would be 1 to
  // 28 % faster here, where a pass takes less than `plan` allows for it
  // (32 of 200 B1 T2048 109 / 87, 8 of 248 B4 T4096 203 / 167); one of 4096 tokens in 8
  // heads is better apart (184 wide 80 / 164).
  const float apart = 34.0f + 0.0255f / 5632 * (float)B * T * W;
  return plan(B, H, T, W / H, true).split.us < apart;
}

hipError_t launch_block_prefill_slices_bf16(const FusedArgs& a, hipStream_t s) {
  const int bw = a.W / a.H;
  if (bw < 128 || bw > 256 || bw % 8 || a.B <= 0 ||
      (int64_t)a.T * a.W * 2 >= (int64_t)0x7fffffff)
    return hipErrorInvalidValue;
  if (a.w_packed &&
      prefill_many_serve(a.B, a.H, a.T, bw, a.gate_branch != nullptr,
                         a.conv_w != nullptr, a.h0 != nullptr))
    return a.gate_branch ? launch_many<true>(a, s) : launch_many<false>(a, s);
  const Plan p = plan(a.B, a.H, a.T, bw, a.gate_branch != nullptr);
  if (a.w_packed)
    return a.gate_branch ? launch_as<true, true>(a, p, s)
                         : launch_as<true, false>(a, p, s);
  return a.gate_branch ? launch_as<false, true>(a, p, s)
                       : launch_as<false, false>(a, p, s);
}

}  // namespace rg
