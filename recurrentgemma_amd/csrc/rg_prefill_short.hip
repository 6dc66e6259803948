// Recurrent core of a prefill in one launch (bf16, 256-wide heads), the form for few
// (row, head) pairs and rows of some hundred tokens: the tiles of a row side by side.
//
// A workgroup of eight waves (two per SIMD) owns 32 channels of one head of one row, for
// the whole row: 8 B x H workgroups.  Per segment of 384 tokens a wave takes every
// eighth tile of 16 tokens, alone from the rows of x to the gates: a tile's 256 input
// channels come in two passes of 128, loaded (eight channels of four rows a lane),
// convolved (every workgroup of a head convolves the same rows again: 42 vector
// instructions per four rows and channel pair) and staged in LDS; 16
// v_mfma_f32_16x16x32_bf16 per pass against the wave's weights give the pre-activations
// of the 32 channels, the gates leave (a, scaled input) per token and channel in LDS.
// Then the workgroup scans the segment as 16 chunks of 24 tokens per channel (chunk
// summaries, a scan over them by lane shifts, replay in place) and writes y, eight
// channels of a token a thread, joined on the way.  Nothing meets at a barrier but the
// ends of the two stages, where the forms for more pairs do at every tile.
// Arithmetic and roundings are those of rg_prefill_teams.hip except for the order in
// which the float32 state is combined.
//
// Bound by vector issue and latencies: a turn of eight tiles takes 3.3 us, 590 vector
// instructions a wave and two waves a SIMD 2.2 of them; launch, weights and one scan 8.
// 3 x 333 tokens, W2560, joined (240 workgroups): slices of 64 channels, 120 workgroups,
// 22.3 us, here 18.6; 1 x 512, in chunks of the row, two launches, 41, here 26.  The
// outputs leaving as two bytes a thread with the join there: 22 and 33.
//
// Replaces the chain Conv1D.forward -> RGLRU.forward of
// recurrentgemma/torch/modules.py:632-643 (layers.py:447-529, 313-365,
// 140-191) for such shapes.
#include "rg_common.h"
#include "rg_internal.h"
#include "rg_row_tiles.h"

namespace rg {
namespace {

using namespace row_tiles;

constexpr int kBW = 256;    // head width
constexpr int kCh = 32;     // output channels per workgroup
constexpr int kSlices = kBW / kCh;
constexpr int kWaves = 8;   // two per SIMD
constexpr int kThreads = kWaves * 64;
constexpr int kTurns = 3;   // of kWaves tiles in a segment
constexpr int kSeg = kTurns * kWaves * kTile;  // 384 tokens
constexpr int kPass = 128;                     // input channels of a pass (two a tile)
constexpr int kRow = 2 * kPass;                // bytes of a staged row
constexpr int kSteps = kBW / 32;               // matrix instructions along k
constexpr int kChunks = kThreads / kCh;        // of a segment in the scan
constexpr int kChunk = kSeg / kChunks;         // 24 tokens each
constexpr int kOut = kSeg * kCh / 8 / kThreads;  // 16-byte outputs of a thread

// Where token t of a segment keeps channel c in ShortLds::a / xn: pairs of tokens fill
// the 64 banks, their four parts of 16 exchanged by the token's group of four, so that
// neither the gate stage (a wave writes 16 channels of tokens 4 g + q, g = 0..3, at
// once) nor the scan (32 channels of two tokens 24 apart) meets a bank twice.
__device__ __forceinline__ int gate_slot(int t, int c) {
  return (t >> 1) * 64 + (((t & 1) * 32 + c) ^ (((t >> 2) & 3) * 16));
}

struct ShortLds {
  // conv output of a pass: row r's 16-byte parts exchanged by r & 7
  unsigned char stage[kWaves][kTile * kRow];
  float a[kSeg * kCh];          // per token and channel: a_t
  float xn[kSeg * kCh];         // ... and the scaled input
  float chunk_p[kChunks][kCh];  // product of a over a chunk
  float chunk_h[kChunks][kCh];  // its state from a zero start,
                                // then the state it starts from
  float carry[kCh];             // state at the segment's start
  f32x4 gates[kCh];             // biases of both gates, inverse decay
  // conv taps of the head's channel pairs, as time pairs (rg_common.h), and biases
  u32x4 taps[kBW / 2];
  f32x2 conv_bias[kBW / 2];
};
static_assert(sizeof(ShortLds) <= 160 * 1024, "one workgroup a CU");

// The wave's weights (256 x 32 per gate, B operands of v_mfma_f32_16x16x32_bf16) live
// in the accumulation registers, all 128 of them, as values that the compiler knows; the
// matrix instructions being inline assembly, it does not count the wait states between
// one and a vector instruction that reads its result: a tile's last four and the wait
// for the results of all are ONE statement.
__device__ __forceinline__ void read_weights(uint32_t at, u32x4 (&w)[2][4]) {
  asm volatile(
      "ds_read_b128 %0, %8\n\t"
      "ds_read_b128 %1, %8 offset:1024\n\t"
      "ds_read_b128 %2, %8 offset:2048\n\t"
      "ds_read_b128 %3, %8 offset:3072\n\t"
      "ds_read_b128 %4, %8 offset:4096\n\t"
      "ds_read_b128 %5, %8 offset:5120\n\t"
      "ds_read_b128 %6, %8 offset:6144\n\t"
      "ds_read_b128 %7, %8 offset:7168\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&a"(w[0][0]), "=&a"(w[0][1]), "=&a"(w[0][2]), "=&a"(w[0][3]), "=&a"(w[1][0]),
        "=&a"(w[1][1]), "=&a"(w[1][2]), "=&a"(w[1][3])
      : "v"(at)
      : "memory");
}
__device__ __forceinline__ void mfma_kept(u32x4 a, u32x4 w, f32x4& acc) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
               : "+v"(acc)
               : "v"(a), "a"(w));
}
__device__ __forceinline__ void mfma_last(u32x4 a, const u32x4 (&w)[4], f32x4 (&acc)[4]) {
  asm volatile(
      "v_mfma_f32_16x16x32_bf16 %0, %4, %5, %0\n\t"
      "v_mfma_f32_16x16x32_bf16 %1, %4, %6, %1\n\t"
      "v_mfma_f32_16x16x32_bf16 %2, %4, %7, %2\n\t"
      "v_mfma_f32_16x16x32_bf16 %3, %4, %8, %3\n\t"
      "s_nop 15\n\t"
      "s_nop 3"
      : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
      : "v"(a), "a"(w[0]), "a"(w[1]), "a"(w[2]), "a"(w[3]));
}

// GELU: y leaves as y * gelu(gate_branch), the join of the recurrent block's two
// branches (recurrentgemma/torch/modules.py:627-628, 644).  PACKED: gate weights in
// operand order (launch_pack_gate_weights), else as the reference lays them out.
template <bool HAS_CONV, bool PACKED, bool GELU>
__global__ void __launch_bounds__(kThreads)
block_prefill_short_bf16_kernel(FusedArgs p) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  ShortLds& lds = *reinterpret_cast<ShortLds*>(lds_raw);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Slice own_slice = slice_of_workgroup<kSlices>();
  const int pair = own_slice.pair, s = own_slice.s;
  if (pair >= p.B * p.H) return;
  const int h = pair % p.H;
  const int b = pair / p.H;
  const int T = p.T;
  const int64_t W = p.W;
  const int c_head = h * kBW;       // first channel of the head
  const int c0 = c_head + s * kCh;  // first channel of this workgroup
  // matrix layout: lane = (g, n); conv layout: eight channels (part n of a pass) of
  // the four rows 4 g .. 4 g + 3
  const int g = lane >> 4;
  const int n = lane & 15;

  // biases and inverse decay of the own channels
  if (tid < kCh) {
    const int c = c0 + tid;
    lds.gates[tid] = f32x4{
        -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[0])[c]),
        -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[1])[c]),
        inverse_decay((-8.0f * kLog2e) *
                      softplus_precise(
                          bf16_bits_to_f32(((const uint16_t*)p.a_param)[c]))),
        0.0f};
  }
  if (HAS_CONV && tid < kBW / 2) {
    const uint16_t* cw = (const uint16_t*)p.conv_w + c_head + 2 * tid;
    uint32_t u[4], w10[2], w32[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = *reinterpret_cast<const uint32_t*>(cw + k * W);
    const uint32_t ub = *reinterpret_cast<const uint32_t*>(
        (const uint16_t*)p.conv_b + c_head + 2 * tid);
    pair_up(u[0], u[1], w10[0], w10[1]);
    pair_up(u[2], u[3], w32[0], w32[1]);
    lds.taps[tid] = u32x4{w10[0], w10[1], w32[0], w32[1]};
    lds.conv_bias[tid] =
        f32x2{__uint_as_float(ub << 16), __uint_as_float(ub & 0xffff0000u)};
  }

  // ---- weights: a wave fetches the 32 k of its number, a lane (g, n) the eight from
  //      8 g on of columns n and 16 + n, which is what that lane of every wave
  //      multiplies; by way of LDS (where the gates' results will live) ----
  u32x4 w[kSteps / 2][2][4];  // [k / 64][k / 32 % 2][2 gate + half of the channels]
  {
    u32x4* const kept = reinterpret_cast<u32x4*>(&lds.a[0]);
    static_assert(sizeof(lds.a) >= 4 * kSteps * 64 * 16, "");
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int gate = i >> 1, half = i & 1;
      if (PACKED) {
        // blocks of 16 k x 32 channels, gates in turn; lane 32 (k / 8) + channel
        v[i] = reinterpret_cast<const u32x4*>(
            p.w_packed)[((int64_t)((h * kSlices + s) * 16 + 2 * wave + (g >> 1)) * 2 +
                         gate) * 64 + 32 * (g & 1) + 16 * half + n];
      } else {
        const uint16_t* src = (const uint16_t*)p.w[gate] + (int64_t)h * kBW * kBW +
                              (32 * wave + 8 * g) * kBW + s * kCh + 16 * half + n;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[i][j] = (uint32_t)src[2 * j * kBW] | (uint32_t)src[(2 * j + 1) * kBW] << 16;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) kept[(wave * 4 + i) * 64 + lane] = v[i];
    __syncthreads();
    const uint32_t at =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)kept +
        16u * (uint32_t)lane;
    static_for<0, kSteps / 2>([&](auto ic) RG_INLINE {
      constexpr int i = decltype(ic)::value;
      read_weights(at + i * 8192u, w[i]);
    });
  }
  const uint32_t row_bytes = 2u * (uint32_t)W;
  const uint32_t seq_bytes = (uint32_t)T * row_bytes;  // < 2^31 (launcher)
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc((const char*)p.x + (int64_t)b * seq_bytes, seq_bytes);
  const bool seg_is64 = p.seg_kind == kSegI64;
  const uint32_t seg_esize = seg_is64 ? 8u : 4u;
  const __amdgpu_buffer_rsrc_t rseg =
      make_rsrc((const char*)p.segpos + (int64_t)b * T * seg_esize,
                (uint32_t)T * seg_esize);

  if (tid < kCh)
    lds.carry[tid] = p.h0 ? p.h0[(int64_t)b * W + c0 + tid] : 0.0f;
  __syncthreads();  // taps and carry written, every wave has read its weights

  unsigned char* const stage = lds.stage[wave];
  // where this lane's row 4 g of a staged pass begins (row 4 g + r: ^ 272 r), and its
  // operand of a pass's first matrix step (step i: ^ 64 i)
  const int put_at = 4 * g * kRow + (n ^ (4 * (g & 1))) * 16;
  const int take_at = n * kRow + (g ^ (n & 7)) * 16;
  // this lane's first row and part (rows before the sequence lie below zero, that is
  // beyond any descriptor, like the rows past its end: zeros)
  const uint32_t lane_at = (uint32_t)(4 * g - 3) * row_bytes + 2u * (c_head + 8 * n);

  const int nseg = (T + kSeg - 1) / kSeg;
  for (int seg = 0; seg < nseg; ++seg) {
    // ---- stage 1: this wave's tiles of the segment, every eighth, a tile's 256 input
    //      channels in two passes of 128 ----
    // Rows 4 g - 3 .. 4 g + 3 of a tile.  The rows of a pass are requested when the
    // pass before it has consumed its own, and arrive while it multiplies.
    u32x4 xr[7];
    Positions positions;
    auto request_rows = [&](int t0, int pass) RG_INLINE {
      const uint32_t at = lane_at + (uint32_t)t0 * row_bytes + 2u * kPass * pass;
#pragma unroll
      for (int r = HAS_CONV ? 0 : 3; r < 7; ++r)
        xr[r] = __builtin_amdgcn_raw_buffer_load_b128(rx, at + r * row_bytes, 0, 0);
    };
    // The conv of a pass's 128 channels into the stage, a channel pair of the lane's
    // four rows at a time (bit j of `starts` is row j - 2 of the tile).
    auto convolve = [&](int pass, uint32_t starts) RG_INLINE {
      asm volatile("" : "+s"(starts));  // (the cuts below are made where they are used)
      // (in place: the outputs of rows 0 .. 3 take the registers of these rows)
      if (HAS_CONV) {
        const int first_tap = fresh(4 * n) + (kPass / 2) * pass;
        auto each_pair = [&](auto&& rows) RG_INLINE {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const u32x4 taps = lds.taps[first_tap + i];
            const f32x2 bias2 = lds.conv_bias[first_tap + i];
            const uint32_t w10[2] = {taps[0], taps[1]}, w32[2] = {taps[2], taps[3]};
            const float bias[2] = {bias2[0], bias2[1]};
            float o[4][2];
            rows(i, w10, w32, bias, o);
#pragma unroll
            for (int r = 0; r < 4; ++r) xr[r + 3][i] = pack_bf16x2(o[r][0], o[r][1]);
          }
        };
        if (__builtin_expect(starts == 0, 1)) {
          each_pair([&](int i, const uint32_t (&w10)[2], const uint32_t (&w32)[2],
                        const float (&bias)[2], float (&o)[4][2]) RG_INLINE {
            uint32_t q[6][2];  // time pairs ending at rows -2 .. 3
            pair_up(xr[0][i], xr[1][i], q[0][0], q[0][1]);
            pair_up(xr[1][i], xr[2][i], q[1][0], q[1][1]);
            pair_up(xr[3][i], xr[4][i], q[3][0], q[3][1]);
            pair_up(xr[5][i], xr[6][i], q[5][0], q[5][1]);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              q[2][e] = __builtin_amdgcn_alignbit(q[3][e], q[1][e], 16);
              q[4][e] = __builtin_amdgcn_alignbit(q[5][e], q[3][e], 16);
            }
            conv4_dot_row_pair(q[0], q[2], q[1], q[3], w10, w32, bias, o[0], o[1]);
            conv4_dot_row_pair(q[2], q[4], q[3], q[5], w10, w32, bias, o[2], o[3]);
          });
        } else {
          const uint32_t near = starts >> (4 * g);  // bit j: row 4 g + j - 2
          each_pair([&](int i, const uint32_t (&w10)[2], const uint32_t (&w32)[2],
                        const float (&bias)[2], float (&o)[4][2]) RG_INLINE {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              // rows r, r - 1, r - 2, r - 3 without what a start cuts off
              const Cuts cut = cuts_of_row(near, r);
              uint32_t p_old[2], p_new[2];
              pair_up(cut.one ? 0u : xr[r + 2][i], xr[r + 3][i], p_new[0], p_new[1]);
              pair_up(cut.three ? 0u : xr[r][i], cut.two ? 0u : xr[r + 1][i], p_old[0],
                      p_old[1]);
              conv4_dot_x2(p_old, p_new, w10, w32, bias, o[r]);
            }
          });
        }
      }
      const int to = fresh(put_at);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<u32x4*>(stage + (to ^ (272 * r))) = xr[r + 3];
    };
    const int first = seg * kSeg + wave * kTile;
    const int end = min(T, (seg + 1) * kSeg);
    if (first < end) {
      positions.request(rseg, seg_is64, first, lane, T);
      request_rows(first, 0);
    }
#pragma unroll 1
    for (int t0 = first; t0 < end; t0 += kWaves * kTile) {
      const int next_t0 = t0 + kWaves * kTile;
      const uint32_t starts = positions.starts(t0, lane, T);
      // pre-activations of tokens t0 .. t0+15: lane (g, n) ends up with channels n and
      // 16 + n of tokens 4 g .. 4 g + 3
      f32x4 acc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = f32x4{0, 0, 0, 0};
      uint32_t own[4];  // conv output of the lane's tokens and channels
      static_for<0, 2>([&](auto pc) RG_INLINE {
        constexpr int pass = decltype(pc)::value;
        convolve(pass, starts);
        // (the rows are consumed: ask for the next pass's now, not earlier:
        // their registers are the same)
        __builtin_amdgcn_sched_barrier(0);
        if (pass == 0) {
          request_rows(t0, 1);
        } else if (next_t0 < end) {
          request_rows(next_t0, 0);
          positions.request(rseg, seg_is64, next_t0, lane, T);
        }
        __builtin_amdgcn_wave_barrier();
        if (pass == (s >> 2)) {
          const int g = fresh(lane) >> 4, n = fresh(lane) & 15;
          // row 4 g's (row 4 g + q: ^ 272 q; channels 16 further: ^ 32)
          const int at = 4 * g * kRow +
                         ((4 * (s & 3) + (n >> 3)) ^ (4 * (g & 1))) * 16 + (n & 7) * 2;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            own[q] = (uint32_t)*reinterpret_cast<const uint16_t*>(
                         stage + (at ^ (272 * q))) |
                     (uint32_t)*reinterpret_cast<const uint16_t*>(
                         stage + (at ^ (272 * q) ^ 32)) << 16;
        }
        u32x4 a[4];
        const int from = fresh(take_at);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          a[i] = *reinterpret_cast<const u32x4*>(stage + (from ^ (64 * i)));
        static_for<0, 4>([&](auto ic) RG_INLINE {
          constexpr int i = decltype(ic)::value;
          if constexpr (pass == 1 && i == 3) {
            mfma_last(a[i], w[2 * pass + i / 2][i & 1], acc);
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) mfma_kept(a[i], w[2 * pass + i / 2][i & 1][j], acc[j]);
          }
        });
        __builtin_amdgcn_wave_barrier();
      });
      // gate arithmetic (layers.py:343-365) of a lane's four tokens -> (a, scaled
      // input) in LDS
      const int g = fresh(lane) >> 4, n = fresh(lane) & 15;
      float av[2][4], xn[2][4];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const f32x4 per_channel = lds.gates[16 * m + n];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float gx = __builtin_amdgcn_rcpf(
              1.0f + __builtin_amdgcn_exp2f(
                         __builtin_fmaf(acc[m][q], -kLog2e, per_channel[0])));
          av[m][q] = __builtin_amdgcn_exp2f(
              gate_exponent(__builtin_amdgcn_exp2f(__builtin_fmaf(
                                acc[2 + m][q], -kLog2e, per_channel[1])),
                            per_channel[2]));
          xn[m][q] = gx * __uint_as_float(m == 0 ? own[q] << 16 : own[q] & 0xffff0000u);
        }
      }
      if (__builtin_expect(starts >> 2 != 0 || t0 + kTile > T, 0)) {
        // document start: forget the state; past the end: identity
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const bool in = t0 + 4 * g + q < T;
            if ((starts >> (4 * g + q + 2)) & 1u) av[m][q] = 0.0f;
            av[m][q] = in ? av[m][q] : 1.0f;
            xn[m][q] = in ? xn[m][q] : 0.0f;
          }
      }
      {
        const int base = (t0 - seg * kSeg) * kCh + 4 * kCh * g + n;
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            // gate_slot(t0 - seg * kSeg + 4 g + q, 16 m + n)
            const int at = base + (q >> 1) * 64 + (((q & 1) * 32 + 16 * m) ^ (16 * g));
            lds.a[at] = av[m][q];
            lds.xn[at] = xn[m][q] * __builtin_amdgcn_sqrtf(
                                        __builtin_fmaf(-av[m][q], av[m][q], 1.0f));
          }
      }
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // ---- stage 2: the recurrence over the segment, 16 chunks per channel ----
    {
      const int tid = fresh((int)threadIdx.x), lane = tid & 63;
      // (the joined branch's rows as the outputs leave, eight channels a thread)
      u32x4 other[kOut];
      const uint32_t out_at = (uint32_t)(seg * kSeg + tid / 4) * row_bytes +
                              2u * (uint32_t)(c0 + 8 * (tid & 3));
      if (GELU) {
        const __amdgpu_buffer_rsrc_t rgate =
            make_rsrc((const char*)p.gate_branch + (int64_t)b * seq_bytes, seq_bytes);
#pragma unroll
        for (int i = 0; i < kOut; ++i)
          other[i] = __builtin_amdgcn_raw_buffer_load_b128(
              rgate, out_at + i * (kThreads / 4) * row_bytes, 0, 0);
      }
      const int ch = tid & (kCh - 1);
      const int chunk = tid / kCh;
      const int i0 = chunk * kChunk;
      const int left = T - (seg * kSeg + i0);
      {
        float pp = 1.0f, hh = 0.0f;
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
          // (the last tile's rows past the end are the identity, those of no tile
          // were never written)
          const int at = gate_slot(i0 + i, ch);
          const float a = lds.a[at], x = lds.xn[at];
          hh = __builtin_fmaf(i < left ? a : 1.0f, hh, i < left ? x : 0.0f);
          pp *= i < left ? a : 1.0f;
        }
        lds.chunk_p[chunk][ch] = pp;
        lds.chunk_h[chunk][ch] = hh;
      }
      __syncthreads();
      chunk_starts(lds.chunk_p, lds.chunk_h, lds.carry, wave, lane);
      __syncthreads();
      // replay, a token's state where its a was; then eight channels of a token a
      // thread, out with 16 bytes
      float hin = lds.chunk_h[chunk][ch];
#pragma unroll
      for (int i = 0; i < kChunk; ++i) {
        const int at = gate_slot(i0 + i, ch);
        hin = __builtin_fmaf(lds.a[at], hin, lds.xn[at]);
        lds.a[at] = hin;
      }
      __syncthreads();
      const __amdgpu_buffer_rsrc_t ry =
          make_rsrc((char*)p.y + (int64_t)b * seq_bytes, seq_bytes);
#pragma unroll
      for (int i = 0; i < kOut; ++i) {
        const float* from = &lds.a[gate_slot(tid / 4 + i * (kThreads / 4), 8 * (tid & 3))];
        const f32x4 lo = *reinterpret_cast<const f32x4*>(from);
        const f32x4 hi = *reinterpret_cast<const f32x4*>(from + 4);
        u32x4 out = {pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]),
                     pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
        if (GELU) {
#pragma unroll
          for (int k = 0; k < 4; ++k) out[k] = gelu_mul_bf16x2(out[k], other[i][k]);
        }
        // (rows past the end are beyond the descriptor)
        buffer_store_16(out, ry, out_at + i * (kThreads / 4) * row_bytes, 0);
      }
    }
    __syncthreads();  // a, xn and the chunk states are free again
  }

  if (p.h_last && tid < kCh) p.h_last[(int64_t)b * W + c0 + tid] = lds.carry[tid];

  if (p.cache_out && tid < kCh) leave_conv_state<uint16_t>(p, b, c0 + tid);
}

template <bool HAS_CONV, bool PACKED, bool GELU>
hipError_t launch_as(const FusedArgs& a, dim3 grid, hipStream_t s) {
  static OncePerDevice once;
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)block_prefill_short_bf16_kernel<HAS_CONV, PACKED, GELU>,
      (int)sizeof(ShortLds));
  if (e != hipSuccess) return e;
  block_prefill_short_bf16_kernel<HAS_CONV, PACKED, GELU>
      <<<grid, kThreads, sizeof(ShortLds), s>>>(a);
  return hipGetLastError();
}

template <bool HAS_CONV, bool PACKED>
hipError_t launch_with(const FusedArgs& a, dim3 grid, hipStream_t s) {
  return a.gate_branch ? launch_as<HAS_CONV, PACKED, true>(a, grid, s)
                       : launch_as<HAS_CONV, PACKED, false>(a, grid, s);
}

}  // namespace

// One round of workgroups, and neither the shortest rows (one pass of
// rg_prefill_slices.hip, which loads its weights without the way through LDS) nor those
// long enough for chunks of the row side by side in two launches.  us, from a graph, the
// other forms / here, joined in brackets: W2560 B1 T65 11 / 11 (11 / 12), T128 11 / 11
// (11 / 12), T200 15 / 14 (16 / 16), T333 20 / 17 (22 / 18), T512 35 / 23 (41 / 26), T768
// 36 / 30 (42 / 32), T900 44 / 38 (54 / 42), T1024 37 / 39 (43 / 42), T1536 39 / 56
// (46 / 61), B3 T333 20 / 18 (22 / 19), T512 36 / 25 (43 / 27), T1024 42 / 41 (48 / 44);
// W4096 B2 T512 35 / 24 (41 / 26); two rounds: W4096 B3 T333 21 / 32 (23 / 34), T512
// 35 / 44 (43 / 49), T768 40 / 56 (47 / 62).  One line with the join and without, so that a
// joined call has the plain one's bits: 961 to 1000 tokens are 37 / 38.5 (44 / 42).  Weights
// as the reference lays them out cost 1.3 here and much more in the other forms, W2560 B1
// T129 28 / 14 (29 / 15), T333 33 / 19 (35 / 20), T512 65 / 26 (73 / 28), T1000 69 / 41 (81 /
// 46), 1 to 32 heads alike: the line is the packed weights'.
bool prefill_short_serves(int B, int H, int T) {
  return (int64_t)B * H * kSlices <= 256 && T > 128 && T <= 1000;
}

hipError_t launch_block_prefill_short_bf16(const FusedArgs& a, hipStream_t s) {
  const int64_t pairs = (int64_t)a.B * a.H;
  if (a.W / a.H != kBW || pairs <= 0 || (pairs + 7) * kSlices > 0x7fffffff ||
      (int64_t)a.T * a.W * 2 >= (int64_t)0x7fffffff)
    return hipErrorInvalidValue;
  const dim3 grid = slices_grid(pairs, kSlices);
  if (a.conv_w)
    return a.w_packed ? launch_with<true, true>(a, grid, s)
                      : launch_with<true, false>(a, grid, s);
  return a.w_packed ? launch_with<false, true>(a, grid, s)
                    : launch_with<false, false>(a, grid, s);
}

}  // namespace rg
