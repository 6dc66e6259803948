// What the bf16 prefill kernels with two teams of waves share: rg_prefill_teams.hip,
// rows or chunks by the workgroup, whose opening says how a block of 32 tokens goes
// through phases M and G, and rg_prefill_relay.hip, blocks dealt out.  Their gate
// arithmetic and what comes before their loops stay written out in either: as functions
// of this header they change what the compiler keeps in which registers (blocks dealt
// out, 20 x 4096 at 4096 wide: 556 -> 585 us), while what is here compiles to the same
// code as before.
#ifndef RG_TWO_TEAMS_H_
#define RG_TWO_TEAMS_H_

#include "rg_common.h"
#include "rg_weight_frags.h"

namespace rg {
namespace two_teams {

constexpr int kBW = 256;   // head width (K and per-gate N)
constexpr int kBT = 32;    // tokens per block
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
// Conv output of a block (the MFMA A operand), bf16, rows padded to 264 elements; a
// ring of three blocks (a block is written over two phases, read over the three after
// them, and a new one starts every second phase).
constexpr int kXcRowBytes = 264 * 2;
constexpr int kXcBlockBytes = kBT * kXcRowBytes;
constexpr int kXcRing = 3;
// Raw x as the memory pipe writes it into LDS: rows of 512 bytes, from four before the
// tokens on.
constexpr int kRawHalo = 4;
constexpr int kRawRowBytes = kBW * 2;
// Per-wave output patch: 16 tokens x 32 channels in bf16, rows padded to 80
// bytes; the second eight rows (the upper lanes') another 64 bytes on, in other
// banks than the first.
constexpr int kPatchStride = 80;
constexpr int kPatchUpper = 8 * kPatchStride + 64;
constexpr int kPatchBytesPerWave = kPatchUpper + 8 * kPatchStride;
// The conv's weights and bias, 32 bytes for each of the head's channel pairs.
constexpr int kConvTabBytes = kBW / 2 * 32;
// Ring of MFMA A operands read ahead of their matrix instruction.
constexpr int kARing = 4;
// Rows of a block that a thread convolves, for two channels.
constexpr int kConvRows = 8;
// How many of a lane's sixteen tokens have their input-gate sigmoid computed
// at the end of phase M, the rest at the top of phase G (measured at B16 T8192
// W4096: 0 -> 755 us, 4 -> 755 us, 8 -> 765 us, 12 -> 777 us a launch), and the
// same for the recurrence gate (any part of it there was slower).
constexpr int kTailXPlain = 0;
constexpr int kTailAPlain = 0;
// ... and with the GELU join in phase G (B8 T4096 W2560 in chunks: 249-256 us for
// 8-16 input-gate and 0-4 recurrence-gate sigmoids here: no difference)
constexpr int kTailXJoined = 16;
constexpr int kTailAJoined = 4;
// Priority of a wave while it issues its matrix instructions (the wave in
// phase G stays at 0 and fills the gaps).
constexpr int kMatrixPriority = 1;

typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint64_t lds_u64;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// ---- width-4 conv -----------------------------------------------------------
struct Conv {  // of a thread's two channels
  uint32_t w10[2], w32[2];
  float bias[2];
};
__device__ __forceinline__ void pair_rows(uint32_t earlier, uint32_t later,
                                          uint32_t (&out)[2]) {
  pair_up(earlier, later, out[0], out[1]);
}

// A thread's kConvRows rows of a block, raw rows -> conv output, in steps that the
// caller spreads between its matrix instructions: the eleven raw rows
// (three of them history), then four row pairs.  The rows are convolved as
// if no document started among them; where one does they are redone with
// the history cut (bit i of `cuts`: row i - 3 of these rows starts a
// document), the same dot products in the same order.  xc_row(i): where the i-th
// goes, in rows behind the first.
struct ConvRows {
  uint32_t raw[kConvRows + 3];
  uint32_t e_prev[2], o_prev[2];
  uint32_t xc_at;
};
__device__ __forceinline__ void conv_load(lds_byte* lds3, uint32_t raw_at,
                                          uint32_t xc_at, ConvRows& cr) {
  cr.xc_at = xc_at;
#pragma unroll
  for (int i = 0; i < kConvRows + 3; ++i)
    cr.raw[i] = *reinterpret_cast<lds_u32*>(lds3 + raw_at + i * kRawRowBytes);
}
template <class XcRow>
__device__ __forceinline__ void conv_pair(lds_byte* lds3, const Conv& conv, ConvRows& cr,
                                          int j, XcRow xc_row) {
  if (j == 0) {
    pair_rows(cr.raw[0], cr.raw[1], cr.o_prev);
    pair_rows(cr.raw[1], cr.raw[2], cr.e_prev);
  }
  uint32_t e[2], o[2];
  pair_rows(cr.raw[3 + 2 * j], cr.raw[4 + 2 * j], e);
  float even[2], odd[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
    o[c] = __builtin_amdgcn_alignbit(e[c], cr.e_prev[c], 16);
  conv4_dot_row_pair(cr.o_prev, o, cr.e_prev, e, conv.w10, conv.w32, conv.bias, even,
                     odd);
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    cr.e_prev[c] = e[c];
    cr.o_prev[c] = o[c];
  }
  *reinterpret_cast<lds_u32*>(lds3 + cr.xc_at + xc_row(2 * j) * kXcRowBytes) =
      pack_bf16x2(even[0], even[1]);
  *reinterpret_cast<lds_u32*>(lds3 + cr.xc_at + xc_row(2 * j + 1) * kXcRowBytes) =
      pack_bf16x2(odd[0], odd[1]);
}
template <class XcRow>
__device__ __forceinline__ void conv_with_cuts(lds_byte* lds3, const Conv& conv,
                                               const ConvRows& cr, uint32_t cuts,
                                               XcRow xc_row) {
  uint32_t r_prev = 0, p1[2] = {0, 0}, p2[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < kConvRows + 3; ++i) {
    const uint32_t r = cr.raw[i];
    if ((cuts >> i) & 1u) {
      r_prev = 0;
      p1[0] = p1[1] = p2[0] = p2[1] = 0;
    }
    uint32_t pt[2];
    pair_rows(r_prev, r, pt);
    if (i >= 3) {
      float o[2];
      conv4_dot_x2(p2, pt, conv.w10, conv.w32, conv.bias, o);
      *reinterpret_cast<lds_u32*>(lds3 + cr.xc_at + xc_row(i - 3) * kXcRowBytes) =
          pack_bf16x2(o[0], o[1]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      p2[c] = p1[c];
      p1[c] = pt[c];
    }
    r_prev = r;
  }
}

}  // namespace two_teams
}  // namespace rg
#endif  // RG_TWO_TEAMS_H_
