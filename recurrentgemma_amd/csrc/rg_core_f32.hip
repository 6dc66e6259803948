// The recurrent core of a short float32 prefill in ONE launch (256-wide
// heads, few rows): width-4 conv -> both gate projections on the bf16 matrix
// instruction, every float32 in three bf16 pieces -> gate activations -> recurrence.
//
// The form of several launches spends most of a small call waiting for launches and
// for each kernel's first loads.  Here one workgroup of eight waves (two per SIMD) owns
// 16 channels of one head of one row for the whole sequence: 16 B x H workgroups.  Per
// segment of 512 tokens a wave takes every eighth tile of 16 tokens (a sequence of up
// to 128 is one tile a wave), and a tile's 256 input channels in four passes of 64:
// rows loaded (four channels of four rows a lane), convolved, cut into pieces and staged
// in LDS (every workgroup of a head convolves the same rows again: 4 multiply-adds per
// element); 24 v_mfma_f32_16x16x32_bf16 per pass against the wave's weights give the
// pre-activations of the 16 channels, the gate arithmetic leaves (a, a-scaled input)
// per token and channel in LDS; then the workgroup scans the segment as 32 chunks of
// 16 tokens per channel (chunk summaries, a scan over the summaries by lane shifts,
// replay) and stores y.
//
// A product is the six products of pieces that weigh most, what is left out below
// 2^-22 of it; the products of the first pieces have an accumulator of their own, the
// others' is 2^-7 times smaller.  Error of y against 64 bits, relative norm, with the
// float32 matrix instruction / now, mean of 16 sets each (inputs as large, a twentieth and
// eight times): 1 x 33 tokens, W4096 9.6e-8 / 8.6e-8, 1 x 200 W2560 and W4096 1.28e-7 /
// 1.22e-7, 1 x 512 1.73e-7 / 1.69e-7, 1 x 1000 2.16e-7 / 2.14e-7; set by set 0.80 to 1.02 of
// what it was, in the mean 0.91 (33 tokens) to 0.99 (1000).  Same conv4() tap
// chain as the other float32 kernels, conv state identical; exp2, reciprocal and
// square root of the gate arithmetic are the hardware's.
//
// us from a graph, on the float32 matrix instruction (which keeps the SIMD's vector
// unit busy: matrix and vector work added up, and four tiles a wave were worked off
// whatever there was of a sequence) / now: W2560 1 x 16 tokens 33.7 / 10, 1 x 128
// 33.7 / 11.6, 1 x 512 35.8 / 27.8, 1 x 1024 66 / 47, 2 x 300 65.6 / 35; W4096 1 x 512
// 36.4 / 30.  A turn of eight tiles takes 5.4 us, launch, weights and scan 6.  Without
// the matrix instructions 24.2 of 27.8, without the cutting 26.5, without the row loads
// 29.2 of 29.7, the reads of a pass all in front of its products 27.6 with no register
// left: bound by the vector instructions (830 a tile and wave, two waves a SIMD) and the
// 0.7 us a turn and SIMD that the LDS port is busy beside them.
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

constexpr int kBW = 256;      // head width
constexpr int kCh = 16;       // output channels per workgroup
constexpr int kSlices = kBW / kCh;
constexpr int kSeg = 512;     // tokens per segment
constexpr int kWaves = 8;     // two per SIMD
constexpr int kThreads = kWaves * 64;
constexpr int kPasses = 4;                 // of a tile's input channels,
constexpr int kPass = kBW / kPasses;       // 64 each
constexpr int kSteps = kBW / 32;           // matrix instructions along k
constexpr int kRow = 2 * kPass;            // bytes of a staged row of one piece
constexpr int kPiece = kTile * kRow;
constexpr int kChunk = 16;                 // tokens per scan chunk
constexpr int kChunks = kSeg / kChunk;     // 32

// Where token t of a segment keeps its 16 channels in CoreF32Lds::a / xn: four
// tokens fill the 64 banks, and which quarter of them a token takes rotates
// with the token's group of 4 and group of 16, so that neither the gate
// stage (a wave writes tokens 4 g + q, g = 0..3, at once) nor the scan (a wave
// reads tokens 16 c + i of four chunks c at once) meets a bank twice.
__device__ __forceinline__ int gate_slot(int t) {
  return (t & ~3) + (((t & 3) + (t >> 2) + (t >> 4)) & 3);
}

struct CoreF32Lds {
  // conv output of a pass, [piece][row][64 channels] in bf16: row r lies in
  // line r ^ (r / 4 & 1), its 16-byte parts exchanged by r & 7
  unsigned char stage[kWaves][3 * kPiece];
  u32x4 w_lo[2][kSteps][64];  // last piece of the weights, operand order
  float a[kSeg][kCh];         // per token and channel: a_t
  float xn[kSeg][kCh];        // ... and the scaled input
  float chunk_p[kChunks][kCh];  // product of a over a chunk
  float chunk_h[kChunks][kCh];  // its state from a zero start,
                                // then the state it starts from
  float carry[kCh];             // state at the segment's start
  f32x4 taps[5][kBW / 4];         // conv taps and bias
};
static_assert(sizeof(CoreF32Lds) <= 160 * 1024, "one workgroup a CU");

// The first two pieces of the wave's weights (256 x 16 per gate, B operands of
// v_mfma_f32_16x16x32_bf16) live in the accumulation registers, all 128 of
// them: with two waves per SIMD a wave has 256 registers, and the other 128 are
// what the rows in flight, the accumulators and the arithmetic need.  The third
// piece, used once a tile where the first is used three times, is read from LDS.
// (Left to the compiler, the accumulators go to the accumulation registers and
// every weight is moved to an ordinary register before its use.)
//
// The matrix instructions being inline assembly, the compiler does not count
// the wait states between one and a vector instruction that reads its result: a
// tile's last two matrix instructions and the wait for the results of all are ONE
// statement.
__device__ __forceinline__ void read_weights(uint32_t at, u32x4& w0, u32x4& w1,
                                             u32x4& w2, u32x4& w3) {
  asm volatile(
      "ds_read_b128 %0, %4\n\t"
      "ds_read_b128 %1, %4 offset:1024\n\t"
      "ds_read_b128 %2, %4 offset:2048\n\t"
      "ds_read_b128 %3, %4 offset:3072\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&a"(w0), "=&a"(w1), "=&a"(w2), "=&a"(w3)
      : "v"(at)
      : "memory");
}
__device__ __forceinline__ void mfma_kept(u32x4 a, u32x4 w, f32x4& acc) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
               : "+v"(acc)
               : "v"(a), "a"(w));
}
__device__ __forceinline__ void mfma_read(u32x4 a, u32x4 w, f32x4& acc) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
               : "+v"(acc)
               : "v"(a), "v"(w));
}
__device__ __forceinline__ void mfma_last(u32x4 a, u32x4 w_x, u32x4 w_a, f32x4& hi_x,
                                          f32x4& hi_a, f32x4& low_x, f32x4& low_a) {
  asm volatile(
      "v_mfma_f32_16x16x32_bf16 %2, %4, %5, %2\n\t"
      "v_mfma_f32_16x16x32_bf16 %3, %4, %6, %3\n\t"
      "s_nop 15\n\t"
      "s_nop 3"
      : "+v"(hi_x), "+v"(hi_a), "+v"(low_x), "+v"(low_a)
      : "v"(a), "v"(w_x), "v"(w_a));
}
__device__ __forceinline__ void mfma_f32(float a, float w, f32x4& acc) {
  asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0"
               : "+v"(acc)
               : "v"(a), "v"(w));
}
// Two conv outputs as three bf16 pieces each: the first cut off, the second rounded, and
// all that is left in the third, which has at most eight bits of it.  Five instructions a
// value; every piece rounded to nearest takes five and a half and leaves out half as much
// of a product.
__device__ __forceinline__ void cut_rows(float a, float b, uint32_t (&piece)[3]) {
  const uint32_t upper = 0x07060302u;  // the upper halves of two registers
  piece[0] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), upper);
  a -= __uint_as_float(__float_as_uint(a) & 0xffff0000u);
  b -= __uint_as_float(__float_as_uint(b) & 0xffff0000u);
  piece[1] = pack_bf16x2(a, b);
  a -= __uint_as_float(piece[1] << 16);
  b -= __uint_as_float(piece[1] & 0xffff0000u);
  piece[2] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), upper);
}
// From here on the pieces of a value hold all of it: the last of its 24 bits is worth
// 2^-133, the least that a bf16 has.  (Below 2^-134, 5e-41, they are zeros.)
constexpr float kExactOwn = 0x1p-110f;

// GELU: y is written as y * gelu(gate_branch), the join of the recurrent
// block's two branches (recurrentgemma/torch/modules.py:627-628, 644).
template <bool HAS_CONV, bool GELU>
__global__ void __launch_bounds__(kThreads) core_f32_small_kernel(FusedArgs p) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  CoreF32Lds& lds = *reinterpret_cast<CoreF32Lds*>(lds_raw);

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
  const int c_head = h * kBW;         // first channel of the head
  const int c0 = c_head + s * kCh;    // first channel of this workgroup
  // matrix layout: lane = (g, n); conv layout: four channels (quad n of a pass)
  // of the four rows 4 g .. 4 g + 3
  const int g = lane >> 4;
  const int n = lane & 15;

  // (the small per-channel loads first, so that they travel together with
  // the weights instead of after them)
  const float bias_x = ((const float*)p.b[0])[c0 + n];
  const float bias_a = ((const float*)p.b[1])[c0 + n];
  // log2 a_t = sigmoid(.) * (-8 log2(e) softplus(a_param))  (layers.py:343-349)
  const float decay2 =
      -8.0f * kLog2e * softplus_precise(((const float*)p.a_param)[c0 + n]);

  // without conv weights x is the conv output already
  constexpr bool has_conv = HAS_CONV;
  if (has_conv && tid < 5 * (kBW / 4)) {
    const int k = tid / (kBW / 4), quad = tid % (kBW / 4);
    const float* src = k < 4 ? (const float*)p.conv_w + k * W : (const float*)p.conv_b;
    lds.taps[k][quad] = *reinterpret_cast<const f32x4*>(src + c_head + 4 * quad);
  }

  // ---- weights: a wave cuts the 32 k of its number, a lane (g, n) the eight from
  //      8 g on of column n, which is what that lane of every wave multiplies ----
  const float* const w_head[2] = {
      (const float*)p.w[0] + (int64_t)h * kBW * kBW + s * kCh,
      (const float*)p.w[1] + (int64_t)h * kBW * kBW + s * kCh};
  u32x4 w_hi[2][kSteps], w_mid[2][kSteps];
  {
    u32x4* const kept = reinterpret_cast<u32x4*>(&lds.a[0][0]);
    static_assert(sizeof(lds.a) + sizeof(lds.xn) >= 4 * kSteps * 64 * 16, "");
    float v[2][8];
#pragma unroll
    for (int gate = 0; gate < 2; ++gate)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[gate][j] = w_head[gate][(32 * wave + 8 * g + j) * kBW + n];
#pragma unroll
    for (int gate = 0; gate < 2; ++gate) {
      u32x4 hi, mid, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t piece[3];
        cut_bf16x2(v[gate][2 * j], v[gate][2 * j + 1], piece);
        hi[j] = piece[0];
        mid[j] = piece[1];
        lo[j] = piece[2];
      }
      kept[((2 * gate + 0) * kSteps + wave) * 64 + lane] = hi;
      kept[((2 * gate + 1) * kSteps + wave) * 64 + lane] = mid;
      lds.w_lo[gate][wave][lane] = lo;
    }
    __syncthreads();
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)kept +
                        16u * (uint32_t)lane;
    static_for<0, 2>([&](auto gc) {
      constexpr int gate = decltype(gc)::value;
      static_for<0, kSteps / 4>([&](auto ic) {
        constexpr int i = 4 * decltype(ic)::value;
        read_weights(at + (2 * gate * kSteps + i) * 1024u, w_hi[gate][i],
                     w_hi[gate][i + 1], w_hi[gate][i + 2], w_hi[gate][i + 3]);
        read_weights(at + ((2 * gate + 1) * kSteps + i) * 1024u, w_mid[gate][i],
                     w_mid[gate][i + 1], w_mid[gate][i + 2], w_mid[gate][i + 3]);
      });
    });
  }
  const uint32_t row_bytes = 4u * (uint32_t)W;
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
  // where this lane's row 4 g of a staged pass begins (row 4 g + r: ^ 144 r), and
  // its operand of a pass's first matrix step (the second: ^ 64)
  const int put_at = g * 4 * kRow + (g & 1) * kRow +
                     ((n >> 1) ^ (4 * (g & 1))) * 16 + (n & 1) * 8;
  const int take_at = (n ^ ((n >> 2) & 1)) * kRow + (g ^ (n & 7)) * 16;
  // this lane's first row and quad (rows before the sequence lie below zero, that
  // is beyond any descriptor, like the rows past its end: zeros)
  const uint32_t lane_at = (uint32_t)(4 * g - 3) * row_bytes + 4u * (c_head + 4 * n);

  const int nseg = (T + kSeg - 1) / kSeg;
  for (int seg = 0; seg < nseg; ++seg) {
    // ---- stage 1: this wave's tiles of the segment, every eighth, a tile's 256
    //      input channels in four passes of 64 ----
    // Rows 4 g - 3 .. 4 g + 3 of a tile.  The rows of a pass are requested when the
    // pass before it has consumed its own, and arrive while it multiplies.
    f32x4 xr[7];
    Positions positions;
    auto request_rows = [&](int t0, int pass) __attribute__((always_inline)) {
      const uint32_t at = lane_at + (uint32_t)t0 * row_bytes + 4u * kPass * pass;
#pragma unroll
      for (int r = has_conv ? 0 : 3; r < 7; ++r)
        xr[r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              rx, at + r * row_bytes, 0, 0));
    };
    // The conv of a pass's 64 channels: put(r, four channels of row 4 g + r) (bit j of
    // `starts` is row j - 2 of the tile).
    auto convolve = [&](int pass, uint32_t starts, auto&& put)
        __attribute__((always_inline)) {
      asm volatile("" : "+s"(starts));  // (the cuts below are made where they are used)
      f32x4 cw[5];
      if (has_conv) {
#pragma unroll
        for (int k = 0; k < 5; ++k) cw[k] = lds.taps[k][(kPass / 4) * pass + n];
      }
      if (__builtin_expect(starts == 0, 1)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = has_conv
                       ? conv4(xr[r + 3][e], xr[r + 2][e], xr[r + 1][e], xr[r][e],
                               cw[0][e], cw[1][e], cw[2][e], cw[3][e], cw[4][e])
                       : xr[r + 3][e];
          put(r, o);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const Cuts cut = cuts_of_row(starts >> (4 * g), r);
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = has_conv ? conv4(xr[r + 3][e], cut.one ? 0.0f : xr[r + 2][e],
                                    cut.two ? 0.0f : xr[r + 1][e],
                                    cut.three ? 0.0f : xr[r][e], cw[0][e], cw[1][e],
                                    cw[2][e], cw[3][e], cw[4][e])
                            : xr[r + 3][e];
          put(r, o);
        }
      }
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
      // both gates' pre-activations of tokens t0 .. t0+15, channels c0 .. +15:
      // lane (g, n) ends up with channel n of tokens 4 g .. 4 g + 3; the products of
      // the first pieces in one accumulator, the five smaller ones in another
      const float b_x = fresh(bias_x), b_a = fresh(bias_a);
      f32x4 hi_x = {b_x, b_x, b_x, b_x}, low_x = {0, 0, 0, 0};
      float own[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      f32x4 hi_a = {b_a, b_a, b_a, b_a}, low_a = {0, 0, 0, 0};
      static_for<0, kPasses>([&](auto pc) __attribute__((always_inline)) {
        constexpr int pass = decltype(pc)::value;
        convolve(pass, starts, [&](int r, f32x4 o) __attribute__((always_inline)) {
          uint32_t p0[3], p1[3];
          cut_rows(o[0], o[1], p0);
          cut_rows(o[2], o[3], p1);
          unsigned char* const to = stage + (put_at ^ (144 * r));
#pragma unroll
          for (int k = 0; k < 3; ++k)
            *reinterpret_cast<u32x2*>(to + k * kPiece) = u32x2{p0[k], p1[k]};
        });
        // (the rows are consumed: ask for the next pass's now, not earlier:
        // their registers are the same)
        __builtin_amdgcn_sched_barrier(0);
        if (pass + 1 < kPasses) {
          request_rows(t0, pass + 1);
        } else if (next_t0 < end) {
          request_rows(next_t0, 0);
          positions.request(rseg, seg_is64, next_t0, lane, T);
        }
        __builtin_amdgcn_wave_barrier();
        // the conv output of the workgroup's own channels, which the gate arithmetic
        // multiplies, put together again: exactly from kExactOwn on
        if (pass == (s >> 2)) {
          const int g = fresh(lane) >> 4, n = fresh(lane) & 15;
          const int own_at = g * 4 * kRow + (g & 1) * kRow +
                             ((2 * (s & 3) + (n >> 3)) ^ (4 * (g & 1))) * 16 +
                             (n & 7) * 2;  // row 4 g's (row 4 g + q: ^ 144 q)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const unsigned char* const from = stage + (own_at ^ (144 * q));
            float piece[3];
#pragma unroll
            for (int k = 0; k < 3; ++k)
              piece[k] = __uint_as_float(
                  (uint32_t)*reinterpret_cast<const uint16_t*>(from + k * kPiece) << 16);
            own[q] = piece[0] + (piece[1] + piece[2]);
          }
        }
        static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
          constexpr int i = 2 * pass + decltype(ic)::value;
          const unsigned char* const from =
              stage + (take_at ^ (64 * decltype(ic)::value));
          const u32x4 hi = *reinterpret_cast<const u32x4*>(from);
          const u32x4 mid = *reinterpret_cast<const u32x4*>(from + kPiece);
          const u32x4 lo = *reinterpret_cast<const u32x4*>(from + 2 * kPiece);
          const u32x4 wx = lds.w_lo[0][i][lane], wa = lds.w_lo[1][i][lane];
          mfma_kept(hi, w_hi[0][i], hi_x);
          mfma_kept(hi, w_hi[1][i], hi_a);
          mfma_kept(hi, w_mid[0][i], low_x);
          mfma_kept(hi, w_mid[1][i], low_a);
          mfma_kept(mid, w_hi[0][i], low_x);
          mfma_kept(mid, w_hi[1][i], low_a);
          mfma_kept(mid, w_mid[0][i], low_x);
          mfma_kept(mid, w_mid[1][i], low_a);
          mfma_kept(lo, w_hi[0][i], low_x);
          mfma_kept(lo, w_hi[1][i], low_a);
          if constexpr (i == kSteps - 1) {
            mfma_last(hi, wx, wa, hi_x, hi_a, low_x, low_a);
          } else {
            mfma_read(hi, wx, low_x);
            mfma_read(hi, wa, low_a);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        __builtin_amdgcn_wave_barrier();
      });
      f32x4 pre_x = hi_x + low_x, pre_a = hi_a + low_a;
      // A piece of an infinity is no number, and a product of pieces may overflow
      // where the product does not: what is not finite is computed again in float32,
      // and so is a conv output whose last digits the third piece cannot hold (zero is
      // none: one less than it is the largest of all).
      float none = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        none = __builtin_fmaf(pre_a[q], 0.0f, __builtin_fmaf(pre_x[q], 0.0f, none));
      uint32_t least = 0xffffffffu;  // of the magnitudes' bits, twice, less one
#pragma unroll
      for (int q = 0; q < 4; ++q)
        least = min(least, (__float_as_uint(own[q]) << 1) - 1u);
      const bool small = least < (__builtin_bit_cast(uint32_t, kExactOwn) << 1) - 1u;
      if (__builtin_expect(__ballot(none != 0.0f || small) != 0, 0)) {
        const float b_x = fresh(bias_x), b_a = fresh(bias_a);
        f32x4 full_x = {b_x, b_x, b_x, b_x}, full_a = {b_a, b_a, b_a, b_a};
        float* const rows = reinterpret_cast<float*>(stage);
        const int g = fresh(lane) >> 4, n = fresh(lane) & 15;
        static_assert(3 * kPiece >= kTile * kPass * 4, "");
#pragma unroll 1
        for (int pass = 0; pass < kPasses; ++pass) {
          request_rows(t0, pass);
          convolve(pass, starts, [&](int r, f32x4 o) __attribute__((always_inline)) {
            *reinterpret_cast<f32x4*>(rows + (4 * g + r) * kPass + 4 * n) = o;
          });
          __builtin_amdgcn_wave_barrier();
          if (pass == (s >> 2)) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              own[q] = rows[(4 * g + q) * kPass + (s & 3) * kCh + n];
          }
#pragma unroll 1
          for (int i = 0; i < kPass / 4; i += 4) {
            float x[4], wx[4], wa[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int k = 4 * (i + j) + g;
              x[j] = rows[n * kPass + k];
              wx[j] = w_head[0][(uint32_t)((kPass * pass + k) * kBW + n)];
              wa[j] = w_head[1][(uint32_t)((kPass * pass + k) * kBW + n)];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              mfma_f32(x[j], wx[j], full_x);
              mfma_f32(x[j], wa[j], full_a);
            }
          }
          __builtin_amdgcn_wave_barrier();
        }
        asm volatile("s_nop 15\n\ts_nop 3" : "+v"(full_x), "+v"(full_a));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (!(fabsf(pre_x[q]) < INFINITY)) pre_x[q] = full_x[q];
          if (!(fabsf(pre_a[q]) < INFINITY)) pre_a[q] = full_a[q];
        }
        if (next_t0 < end) request_rows(next_t0, 0);
      }
      // gate arithmetic (layers.py:343-365) of a lane's four tokens -> (a, scaled
      // input) in LDS
      const int g = fresh(lane) >> 4, n = fresh(lane) & 15;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = 4 * g + q;
        const int t = t0 + r;
        // (the hardware's exp2, reciprocal and square root, about 1 ulp each,
        // where the other float32 kernels call expf, divide and call sqrtf: a
        // quarter of the instructions; an argument's rounding before exp2
        // costs |argument| x 6e-8 of relative error where the result is far
        // from 1 and nothing where it is near: two orders of magnitude inside
        // the 1e-5 bar)
        const float gate_x =
            __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-kLog2e * pre_x[q]));
        const float gate_a =
            __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-kLog2e * pre_a[q]));
        const float log2_a = gate_a * decay2;
        float a = __builtin_amdgcn_exp2f(log2_a);
        float mult = __builtin_amdgcn_sqrtf(
            1.0f - __builtin_amdgcn_exp2f(log2_a + log2_a));
        if ((starts >> (r + 2)) & 1u) {  // document start: forget the state
          a = 0.0f;
          mult = 1.0f;
        }
        float xn = (own[q] * gate_x) * mult;
        if (t >= T) {  // past the end: identity
          a = 1.0f;
          xn = 0.0f;
        }
        const int slot = gate_slot(t - seg * kSeg);
        lds.a[slot][n] = a;
        lds.xn[slot][n] = xn;
      }
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // ---- stage 2: the recurrence over the segment, 32 chunks per channel ----
    {
      const int tid = fresh(threadIdx.x), lane = tid & 63;
      const int ch = tid & (kCh - 1);
      const int chunk = tid >> 4;
      const int i0 = chunk * kChunk;
      // (chunks past the end hold nothing: the identity)
      const int left = T - (seg * kSeg + i0);
      {
        float pp = 1.0f, hh = 0.0f;
        if (left > 0)
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
          const float a = lds.a[gate_slot(i0 + i)][ch];
          hh = __builtin_fmaf(a, hh, lds.xn[gate_slot(i0 + i)][ch]);
          pp *= a;
        }
        lds.chunk_p[chunk][ch] = pp;
        lds.chunk_h[chunk][ch] = hh;
      }
      __syncthreads();
      chunk_starts(lds.chunk_p, lds.chunk_h, lds.carry, wave, lane);
      __syncthreads();
      float hin = lds.chunk_h[chunk][ch];
      const int64_t y_at = ((int64_t)b * T + seg * kSeg + i0) * W + c0 + ch;
      float* y = (float*)p.y + y_at;
      float other[kChunk];  // GELU: the other branch at this thread's tokens
      if (GELU) {
        const float* gb = (const float*)p.gate_branch + y_at;
#pragma unroll
        for (int i = 0; i < kChunk; ++i)
          other[i] = i < left ? gb[(int64_t)i * W] : 0.0f;
      }
      if (left > 0)
#pragma unroll
      for (int i = 0; i < kChunk; ++i) {
        hin = __builtin_fmaf(lds.a[gate_slot(i0 + i)][ch], hin,
                             lds.xn[gate_slot(i0 + i)][ch]);
        if (i < left)
          y[(int64_t)i * W] = GELU ? gelu_mul_f32(hin, other[i]) : hin;
      }
    }
    __syncthreads();  // a, xn and the chunk states are free again
  }

  if (p.h_last && tid < kCh) p.h_last[(int64_t)b * W + c0 + tid] = lds.carry[tid];

  if (p.cache_out && tid < kCh) leave_conv_state<float>(p, b, c0 + tid);
}

}  // namespace

// Shapes this kernel is for: float32, 256-wide heads, at most 32 (row, head)
// pairs (16 workgroups each), rows that fit 31-bit byte offsets.
bool core_f32_small_serves(int B, int T, int W, int H) {
  return W % H == 0 && W / H == kBW && (int64_t)B * H <= 32 &&
         (int64_t)T * W * 4 < (int64_t)0x7fffffff;
}

template <bool HAS_CONV, bool GELU>
static hipError_t launch_core_f32_small_as(const FusedArgs& a, dim3 grid,
                                           hipStream_t s) {
  static OncePerDevice once;
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)core_f32_small_kernel<HAS_CONV, GELU>,
      (int)sizeof(CoreF32Lds));
  if (e != hipSuccess) return e;
  core_f32_small_kernel<HAS_CONV, GELU>
      <<<grid, kThreads, sizeof(CoreF32Lds), s>>>(a);
  return hipGetLastError();
}

hipError_t launch_core_f32_small(const FusedArgs& a, hipStream_t s) {
  const dim3 grid = slices_grid((int64_t)a.B * a.H, kSlices);
  if (a.conv_w)
    return a.gate_branch ? launch_core_f32_small_as<true, true>(a, grid, s)
                         : launch_core_f32_small_as<true, false>(a, grid, s);
  return a.gate_branch ? launch_core_f32_small_as<false, true>(a, grid, s)
                       : launch_core_f32_small_as<false, false>(a, grid, s);
}

}  // namespace rg
