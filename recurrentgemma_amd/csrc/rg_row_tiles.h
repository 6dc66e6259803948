// What the prefill kernels share that deal the tiles of 16 tokens of a row to the waves
// of a workgroup and then scan a segment of them (rg_prefill_short.hip, rg_core_f32.hip):
// which slice of which (row, head) pair a workgroup has, document starts, the states that
// the chunks of a segment start from, the conv state that is left.
#ifndef RG_ROW_TILES_H_
#define RG_ROW_TILES_H_

#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace row_tiles {

#define RG_INLINE __attribute__((always_inline))

constexpr int kTile = 16;  // tokens per matrix tile

// A value that nothing is worked out from ahead of a loop: what is worked out from it is
// worked out again where it is used, instead of being kept in registers.
template <class V>
__device__ __forceinline__ V fresh(V v) {
  asm volatile("" : "+v"(v));
  return v;
}
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// Which pair and which of its SLICES a workgroup has.  Workgroups go to the eight XCDs in
// turn (linear id modulo 8), each with an L2 of its own: the workgroups of a pair, which
// read the same rows and one head's weights, are dealt to ONE of them (pair p runs on XCD
// p % 8; the grid is whole rounds of eight pairs and the surplus exits).
struct Slice {
  int pair, s;
};
template <int SLICES>
__device__ __forceinline__ Slice slice_of_workgroup() {
  const int xcd = blockIdx.x & 7;
  const int in_xcd = blockIdx.x >> 3;
  return {(in_xcd / SLICES) * 8 + xcd, in_xcd % SLICES};
}
inline dim3 slices_grid(int64_t pairs, int slices) {
  return dim3((unsigned)((pairs + 7) / 8 * 8 * slices));
}

// Positions of rows t0 - 2 .. t0 + 15 of a row of T (lane j looks at row t0 - 2 + j),
// requested ahead, and the document starts among them (bit j of the result; rows before
// the row or past its end: no start).
struct Positions {
  uint32_t lo = 1, hi = 0;
  __device__ __forceinline__ static bool in_row(int t, int lane, int T) {
    return lane < kTile + 2 && t >= 0 && t < T;
  }
  __device__ __forceinline__ void request(const __amdgpu_buffer_rsrc_t& rseg, bool is64,
                                          int t0, int lane, int T) {
    const int t = t0 - 2 + lane;
    const uint32_t off =
        in_row(t, lane, T) ? (uint32_t)t * (is64 ? 8u : 4u) : kBufferOutOfRange;
    lo = __builtin_amdgcn_raw_buffer_load_b32(rseg, off, 0, 0);
    hi = __builtin_amdgcn_raw_buffer_load_b32(rseg, is64 ? off + 4u : kBufferOutOfRange,
                                              0, 0);
  }
  __device__ __forceinline__ uint32_t starts(int t0, int lane, int T) const {
    return (uint32_t)__ballot(in_row(t0 - 2 + lane, lane, T) && (lo | hi) == 0u);
  }
};

// Tap k of a row reads the row k before it, which counts only if no document starts in
// between or at the row itself.  near: starts >> (first of a lane's rows), r: which of
// them.
struct Cuts {
  bool one, two, three;  // whether taps 1, 2 and 3 are cut off
};
__device__ __forceinline__ Cuts cuts_of_row(uint32_t near, int r) {
  Cuts c;
  c.one = (near >> (r + 2)) & 1u;
  c.two = c.one || ((near >> (r + 1)) & 1u);
  c.three = c.two || ((near >> r) & 1u);
  return c;
}

// The state every chunk of a segment starts from: a scan over the chunk summaries -- p
// the product of a over a chunk, h its state from a zero start -- with the operator of
// recurrentgemma/jax/scan.py:161-187, by lane shifts inside a wave (lane = 64 / CHUNKS x
// chunk + channel; a wave takes 64 / CHUNKS of the CH channels), left where the chunk's
// own summary was; and the state behind the segment in carry.
template <int CHUNKS, int CH>
__device__ __forceinline__ void chunk_starts(const float (&p)[CHUNKS][CH],
                                             float (&h)[CHUNKS][CH], float (&carry_)[CH],
                                             int wave, int lane) {
  constexpr int kWide = 64 / CHUNKS;
  const int sc = lane / kWide;                        // chunk
  const int sch = kWide * wave + (lane & (kWide - 1));  // channel
  float sp = p[sc][sch], sh = h[sc][sch];
#pragma unroll
  for (int d = 1; d < CHUNKS; d *= 2) {
    const float pp = __shfl_up(sp, kWide * d, 64);
    const float hp = __shfl_up(sh, kWide * d, 64);
    if (sc >= d) {
      sh = __builtin_fmaf(sp, hp, sh);
      sp *= pp;
    }
  }
  // (sp, sh): chunks 0 .. sc from a zero state; the state after chunk sc is sp * carry +
  // sh, and chunk sc starts from its neighbour's
  const float carry = carry_[sch];
  const float after = __builtin_fmaf(sp, carry, sh);
  const float before = __shfl_up(after, kWide, 64);
  h[sc][sch] = sc == 0 ? carry : before;
  if (sc == CHUNKS - 1) carry_[sch] = after;
}

// Masked conv state of channel c of row b: rows T-3..T-1 of x, each zeroed if a document
// starts in a later position of the row; rows before the sequence start are zero.
template <class E>
__device__ __forceinline__ void leave_conv_state(const FusedArgs& p, int b, int c) {
  const int T = p.T;
  const int64_t W = p.W;
  E* cache = (E*)p.cache_out + (int64_t)b * 3 * W + c;
  bool later_start = false;
#pragma unroll
  for (int kk = 2; kk >= 0; --kk) {
    const int t = T - 3 + kk;
    E v = 0;
    if (t >= 0 && !later_start) v = ((const E*)p.x)[((int64_t)b * T + t) * W + c];
    cache[(int64_t)kk * W] = v;
    if (t >= 0 && is_doc_start(p.segpos, p.seg_kind, (int64_t)b * T + t))
      later_start = true;
  }
}

}  // namespace row_tiles
}  // namespace rg

#endif  // RG_ROW_TILES_H_
