// Linear layers of the residual stack for a handful of rows (one decode step
// of a batch of at most 64 sequences): out[M, N] = x[M, K] @ W^T + bias, bf16
// with fp32 accumulation.  These are torch.nn.Linear / Einsum calls in the
// reference (recurrentgemma/torch/modules.py:579-601 linear_y / linear_x /
// linear_out, :711-721 ffw_up / ffw_down, :334-352 the attention projections);
// with M <= 64 each is one pass over its weight matrix and nothing else, so the
// kernel is built around streaming W:
//  * W is repacked once (linear_pack_kernel) into the operand order of
//    v_mfma_f32_32x32x16_bf16: block (tile, k-step) of 1 KB holds, for lane
//    l = 32 g + r, the eight values W[32 tile + r, 16 kstep + 8 g .. +8], so a
//    wave reads its 32 weight rows as one contiguous stream, 1 KB per
//    instruction.  (Reading the row-major matrix directly touches 32 cache
//    lines per instruction and ran at a quarter of the speed.)
//  * A workgroup owns NT tiles of 32 weight rows; its waves split K in chunks
//    of 64 and add their partial sums through LDS at the end.  x (at most
//    64 x K, L2 resident) is staged by each wave for its own chunks: 64 rows
//    x 128 B coalesced from global, through a wave-private LDS tile, into the
//    B-operand fragments.
//  * Few weight rows (N / 32 tiles well below the number of CUs) and a long K:
//    the grid also splits K (gridDim.y), every workgroup writes its fp32
//    partial sums, and linear_finish_kernel adds them in a fixed order, so the
//    result does not depend on which workgroup ran first.
// Epilogues: bias; bias then residual add (two roundings, like the separate
// add of the reference); gelu(gate) * up for the paired rows of the MLP's
// stacked up-projection (modules.py:752-757).
#include "rg_common.h"
#include "rg_internal.h"
#include "rg_norm_row.h"

namespace rg {
namespace {

union Frag {
  u32x4 u;
  bf16x8 v;
};

constexpr int kXStride = 72;  // elements per staged x row: 64 + 8 of padding
constexpr int kWaves = 8;
// of buffer instructions (gfx950)
constexpr int kAgentScope = 16, kNonTemporal = 2;

// LDS of a wave: its x tile (whole blocks of 32 rows) or its sums.
__host__ __device__ constexpr int wave_lds_bytes(int nt, int blocks) {
  const int sums = nt * blocks * 4096, x = 32 * blocks * kXStride * 2;
  return sums > x ? sums : x;
}

enum LinearMode { kStore = 0, kGeluPair = 1, kPartial = 2 };

__device__ __forceinline__ void unpack4(u32x2 b, float (&v)[4]) {
  v[0] = __uint_as_float(b[0] << 16);
  v[1] = __uint_as_float(b[0] & 0xffff0000u);
  v[2] = __uint_as_float(b[1] << 16);
  v[3] = __uint_as_float(b[1] & 0xffff0000u);
}

// Where column n of the result lives: the output is [G][M][gw] with gw = N / G
// (G = 1: plain [M, N]).
__device__ __forceinline__ size_t out_index(int m, int n, int M, int gw) {
  const int grp = n / gw;
  return ((size_t)grp * M + m) * gw + (n - grp * gw);
}

// From the waves' accumulators to the layer's outputs: the sums over K meet in LDS, then
// the epilogue.  block: which NT tiles of weight rows or, HALF, which half of a tile.
template <int NT, int MODE, int XR, bool HALF>
__device__ __forceinline__ void add_up_and_store(
    const LinearArgs& p, unsigned char* const smem, const int wave, const int lane,
    const int block, const f32x16 (&acc)[NT][XR > 32 ? 2 : 1]) {
  constexpr int kMB = XR > 32 ? 2 : 1;
  constexpr int kWaveLds = wave_lds_bytes(NT, kMB);
  const int M = p.M;
  // the waves' partial sums meet in LDS (each wave's region is its own x tile)
  float* mine = reinterpret_cast<float*>(smem + (size_t)wave * kWaveLds);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < kMB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        mine[((t * kMB + m) * 16 + i) * 64 + lane] = acc[t][m][i];
  lds_barrier();
  const float* red = reinterpret_cast<const float*>(smem);
  // sum of accumulator registers 4 q .. 4 q + 3 of (tile t, half m, lane l):
  // result rows 32 m + l % 32, weight rows 32 t + 8 q + 4 (l / 32) + 0..3
  auto gather = [&](int t, int m, int q, int l, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = 0.0f;
    for (int wv = 0; wv < kWaves; ++wv) {
      const float* src = red + (size_t)wv * (kWaveLds / 4) +
                         ((t * kMB + m) * 16 + q * 4) * 64 + l;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += src[i * 64];
    }
  };
  const uint16_t* bias = reinterpret_cast<const uint16_t*>(p.bias);
  uint16_t* out = reinterpret_cast<uint16_t*>(p.out);
  if (MODE == kGeluPair) {
    // tile 0 = 32 rows of the gate half, tile 1 = the same rows of the up half
    static_assert(MODE != kGeluPair || NT == 2, "pairs need two tiles");
    const int half = p.N / 2;
    for (int qd = threadIdx.x; qd < kMB * 4 * 64; qd += kWaves * 64) {
      const int l = qd & 63, q = (qd >> 6) & 3, m = qd >> 8;
      const int row = 32 * m + (l & 31);
      const int col = block * 32 + 8 * q + 4 * (l >> 5);
      if (row >= M) continue;
      float gate[4], up[4];
      gather(0, m, q, l, gate);
      gather(NT - 1, m, q, l, up);
      if (bias) {
        float bg[4], bu[4];
        unpack4(*reinterpret_cast<const u32x2*>(bias + col), bg);
        unpack4(*reinterpret_cast<const u32x2*>(bias + half + col), bu);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          gate[i] += bg[i];
          up[i] += bu[i];
        }
      }
      const u32x2 ov = {gelu_mul_bf16x2(pack_bf16x2(up[0], up[1]),
                                        pack_bf16x2(gate[0], gate[1])),
                        gelu_mul_bf16x2(pack_bf16x2(up[2], up[3]),
                                        pack_bf16x2(gate[2], gate[3]))};
      *reinterpret_cast<u32x2*>(out + (size_t)row * half + col) = ov;
    }
    return;
  }
  static_assert(!HALF || (NT == 1 && MODE == kStore), "");
  constexpr int kQuads = HALF ? 2 : 4;  // of 8 weight rows
  for (int qd = threadIdx.x; qd < NT * kMB * kQuads * 64; qd += kWaves * 64) {
    const int l = qd & 63, m = qd / (64 * kQuads) % kMB;
    const int q = (qd >> 6) % kQuads + (HALF ? (block & 1) * 2 : 0);
    const int t = qd / (64 * kQuads) / kMB;
    const int row = 32 * m + (l & 31);
    const int col = (HALF ? block >> 1 : block * NT + t) * 32 + 8 * q + 4 * (l >> 5);
    if (row >= M) continue;
    float v[4];
    gather(t, m, q, l, v);
    if (MODE == kPartial) {
      const f32x4 o = {v[0], v[1], v[2], v[3]};
      *reinterpret_cast<f32x4*>(p.partial +
                                ((size_t)blockIdx.y * M + row) * p.N + col) = o;
      continue;
    }
    if (bias) {
      float b[4];
      unpack4(*reinterpret_cast<const u32x2*>(bias + col), b);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += b[i];
    }
    const size_t at = out_index(row, col, M, p.group_width);
    if (p.residual) {
      float res[4];
      unpack4(*reinterpret_cast<const u32x2*>(
                  reinterpret_cast<const uint16_t*>(p.residual) + at), res);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = round_to_bf16(v[i]) + res[i];
    }
    const u32x2 ov = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    *reinterpret_cast<u32x2*>(out + at) = ov;
  }
}

// XR: rows of x that are loaded and staged (M rounded up to 16, 32 or 64).
// Every workgroup draws all of x beside its weights: 64 rows are twice the
// bytes of one tile's weights, whether the rows exist or not.
// BESIDE: the grid goes on behind the layer's workgroups with kCopiers that copy
// p.copy_items: what the next launch reads while it overwrites the original.
constexpr int kCopiers = 16;
__device__ __forceinline__ void copy_beside(const LinearArgs& p) {
  const u32x4* from = reinterpret_cast<const u32x4*>(p.copy_from);
  u32x4* to = reinterpret_cast<u32x4*>(p.copy_to);
  constexpr int64_t step = kCopiers * kWaves * 64;
  for (int64_t i = (int64_t)(gridDim.x - 1 - blockIdx.x) * (kWaves * 64) + threadIdx.x;
       i < p.copy_items; i += step)
    to[i] = from[i];
}

// HALF: a workgroup has half a tile of weight rows (the matrix instructions run with zeros
// in place of the others, which gives the same bits).
template <int NT, int MODE, int XR, bool BESIDE, bool HALF>
__global__ void __launch_bounds__(kWaves * 64)
linear_rows_kernel(LinearArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  if (BESIDE && blockIdx.x >= gridDim.x - kCopiers) {
    copy_beside(p);
    return;
  }
  if (MODE == kPartial && p.clear && blockIdx.x + blockIdx.y == 0 && threadIdx.x < kNormFlags)
    p.clear[threadIdx.x] = 0;
  constexpr int kLoads = XR / 8;          // of x per chunk
  constexpr int kMB = XR > 32 ? 2 : 1;    // blocks of 32 result rows
  constexpr int kWaveLds = wave_lds_bytes(NT, kMB);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, g = lane >> 5;
  const int M = p.M, K = p.K;
  const int chunks = K / 64;
  // this workgroup's slice of K, then this wave's
  const int per_wg = (chunks + (int)gridDim.y - 1) / (int)gridDim.y;
  const int wg0 = blockIdx.y * per_wg, wg1 = min(chunks, wg0 + per_wg);
  const int per = (max(wg1 - wg0, 0) + kWaves - 1) / kWaves;
  const int c0 = wg0 + wave * per;
  const int c1 = min(wg1, c0 + per);
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem + (size_t)wave * kWaveLds);

  // x chunk = XR rows x 128 B; load j covers rows 8 j + lane / 8 (rows >= M
  // repeat row M - 1, rows >= XR of the tile hold what LDS held: their results
  // are never stored)
  const int xrow = lane >> 3, xseg = lane & 7;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(p.x);
  const uint16_t* xg[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j)
    xg[j] = x + (size_t)min(8 * j + xrow, M - 1) * K + 8 * xseg;
  const u32x4* wg[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    wg[t] = reinterpret_cast<const u32x4*>(p.w_packed) +
            ((size_t)((HALF ? blockIdx.x >> 1 : blockIdx.x) * NT + t) * (K / 16)) * 64 +
            lane;
  // (the other half's lanes lie outside the descriptor: zeros, and nothing is fetched)
  const __amdgpu_buffer_rsrc_t tile_rows =
      make_rsrc(wg[0] - lane, HALF ? (uint32_t)K * 64u : 0u);
  const uint32_t in_tile =
      (r >> 4) == (int)(blockIdx.x & 1) ? 16u * (uint32_t)lane : kBufferOutOfRange;

  f32x16 acc[NT][kMB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < kMB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][m][i] = 0.0f;

  u32x4 xr[kLoads];
  Frag wq[2][NT][4];
  auto load_chunk = [&](int c, int slot) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      xr[j] = *reinterpret_cast<const u32x4*>(xg[j] + (size_t)c * 64);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        wq[slot][t][k].u =
            HALF ? __builtin_amdgcn_raw_buffer_load_b128(
                       tile_rows, in_tile + (uint32_t)(c * 4 + k) * 1024u, 0, kNonTemporal)
                 : __builtin_nontemporal_load(wg[t] + (size_t)(c * 4 + k) * 64);
  };
  auto body = [&](int slot, int c, bool more) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      *reinterpret_cast<u32x4*>(xs + (8 * j + xrow) * kXStride + 8 * xseg) =
          xr[j];
    Frag xf[4][kMB];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int m = 0; m < kMB; ++m)
        xf[k][m].u = *reinterpret_cast<const u32x4*>(
            xs + (32 * m + r) * kXStride + 16 * k + 8 * g);
    if (more) load_chunk(c + 1, slot ^ 1);
    // (the next chunk's loads stay in front of this one's products)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < kMB; ++m)
          acc[t][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              wq[slot][t][k].v, xf[k][m].v, acc[t][m], 0, 0, 0);
  };
  if (c0 < c1) {
    load_chunk(c0, 0);
    int c = c0;
    for (; c + 2 < c1; c += 2) {
      body(0, c, true);
      body(1, c + 1, true);
    }
    // The last one or two: nothing is loaded behind them.  (A load of the last chunk
    // once more, as an even number of chunks a wave used to have it, is an eighth of
    // the weights at K 4096: us a layer, with / without it, N 8192 at 1, 16, 32, 64
    // rows 15.1 / 14.5, 15.5 / 14.4, 16.7 / 15.4, 19.7 / 18.5; N 24576 in pairs
    // 47.5 / 44; K 2048, N 2560 6.6 / 6.0; odd numbers the same.  More chunks on their
    // way, 3 to 5 of them, are no faster: a CU takes about 40 GB/s whatever waits.)
    if (c + 1 < c1) {
      body(0, c, true);
      body(1, c + 1, false);
    } else {
      body(0, c, false);
    }
  }

  add_up_and_store<NT, MODE, XR, HALF>(p, smem, wave, lane, blockIdx.x, acc);
}

// The norm in front of such layers and the layers as one launch: what a decode step has
// twice in a block.  As launches of their own the norm is 2.5 us of launch and 2 of
// latencies in which nothing else happens, and the layer's first weights are asked for
// behind it.  Here the first M workgroups norm a row each (of what the layer before left
// as partial sums), while the others have all of their weights on their way -- the CPW
// chunks of 64 that a wave has of K, in registers -- and wait for the rows, which the norms'
// workgroups report in a.flags.  Rows and flags are written and read at agent
// scope (a row's stores have arrived before its flag is stored): no fence, which cost 0.3
// to 0.7 us.
// Every wait ends: a workgroup that has looked `patience` times in vain (the norms'
// workgroups, the first of the grid, are not running) norms all rows itself, which writes
// the same bytes once more.
// What bounds it: launch, norm, stores, flag, loads of x one behind the other, 9 us, and
// from 12 MB or so of weights on those.  us a norm and layer, K 2560, replayed from a graph
// over 16 sets of weights, two launches / one: N 5120 at 1, 16, 32 rows 9.9 / 7.9, 11.7 /
// 8.9, 13.4 / 10.3; N 3072 10.3 / 7.9, 11.6 / 8.7, 12.7 / 9.9; pairs of N 15360 18.8 /
// 16.2, 18.1 / 16.5, 19.6 / 18.6.
template <int NT, int MODE, int XR, int CPW, bool BESIDE>
__global__ void __launch_bounds__(kWaves * 64)
linear_rows_normed_kernel(NormedLinearArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float norm_sums[4];
  __shared__ int all_there;
  const LinearArgs& p = a.layer;
  const int M = p.M;
  const int tid = threadIdx.x;
  constexpr int K = CPW * kWaves * 64;
  const auto norm_row = [&](int row) {
    PartialRows part;
    part.sums = reinterpret_cast<const f32x4*>(a.sums);
    part.slices = a.slices;
    part.slice_stride = (int64_t)M * K / 4;
    part.bias = reinterpret_cast<const u32x4*>(a.bias);
    const u32x4* const scale = reinterpret_cast<const u32x4*>(a.scale);
    u32x4* const sum_out = reinterpret_cast<u32x4*>(a.sum_out);
    u32x4* const out = reinterpret_cast<u32x4*>(a.normed);
    if (a.addend)
      rms_norm_row<true, true, true>(tid, row, norm_sums, nullptr, part,
                                     reinterpret_cast<const u32x4*>(a.addend), scale,
                                     sum_out, out, K / 8, 1.0f / (float)K, a.eps);
    else
      rms_norm_row<false, true, true>(tid, row, norm_sums, nullptr, part, nullptr, scale,
                                      sum_out, out, K / 8, 1.0f / (float)K, a.eps);
    // (the agent-scope stores have arrived when they are counted)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  if ((int)blockIdx.x < M) {
    if (tid >= 256) return;
    norm_row(blockIdx.x);
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(a.flags + blockIdx.x, 1u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  if (BESIDE && blockIdx.x >= gridDim.x - kCopiers) {
    copy_beside(p);
    return;
  }
  const int block = blockIdx.x - M;
  constexpr int kLoads = XR / 8;
  constexpr int kMB = XR > 32 ? 2 : 1;
  constexpr int kWaveLds = wave_lds_bytes(NT, kMB);
  // chunks of x on their way beside the weights
  constexpr int kAhead = XR == 16 ? (NT == 1 ? CPW : 3) : XR == 32 ? 2 : 1;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r = lane & 31, g = lane >> 5;
  const int c0 = wave * CPW;
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem + (size_t)wave * kWaveLds);
  const u32x4* wg[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    wg[t] = reinterpret_cast<const u32x4*>(p.w_packed) +
            ((size_t)(block * NT + t) * (K / 16) + c0 * 4) * 64 + lane;
  Frag wq[CPW][NT][4];
  auto load_weights = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        wq[c][t][k].u = __builtin_nontemporal_load(wg[t] + (c * 4 + k) * 64);
  };
#pragma unroll
  for (int c = 0; c < CPW; ++c) load_weights(c);
  __builtin_amdgcn_sched_barrier(0);

  // ---- the rows ------------------------------------------------------------------
  if (wave == 0) {
    int polls = 0;
    bool there = false;
    for (;;) {
      uint32_t flag = 1;
      if (lane < M)
        flag = __hip_atomic_load(a.flags + lane, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      there = __all(flag != 0);
      if (there || ++polls > a.patience) break;
    }
    if (lane == 0) all_there = there;
  }
  lds_barrier();
  if (__builtin_expect(!all_there, 0)) {
    for (int row = 0; row < M; ++row) {
      if (tid < 256)
        norm_row(row);
      else
        __syncthreads();  // (the norm's one)
      __syncthreads();
    }
    // (once more: kept across the norm they are registers too many)
#pragma unroll
    for (int c = 0; c < CPW; ++c) load_weights(c);
  }

  const int xrow = lane >> 3, xseg = lane & 7;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, (uint32_t)M * K * 2u);
  u32x4 xr[kAhead][kLoads];
  // (rows past the last read as zeros)
  auto load_x = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      xr[c % kAhead][j] = __builtin_amdgcn_raw_buffer_load_b128(
          rx, (uint32_t)((8 * j + xrow) * K + (c0 + c) * 64 + 8 * xseg) * 2u, 0,
          kAgentScope);
  };
  f32x16 acc[NT][kMB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < kMB; ++m)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][m][i] = 0.0f;
#pragma unroll
  for (int c = 0; c < kAhead; ++c) load_x(c);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < CPW; ++c) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      *reinterpret_cast<u32x4*>(xs + (8 * j + xrow) * kXStride + 8 * xseg) =
          xr[c % kAhead][j];
    Frag xf[4][kMB];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int m = 0; m < kMB; ++m)
        xf[k][m].u = *reinterpret_cast<const u32x4*>(
            xs + (32 * m + r) * kXStride + 16 * k + 8 * g);
    if (c + kAhead < CPW) load_x(c + kAhead);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < kMB; ++m)
          acc[t][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              wq[c][t][k].v, xf[k][m].v, acc[t][m], 0, 0, 0);
  }
  add_up_and_store<NT, MODE, XR, false>(p, smem, wave, lane, block, acc);
}

// Sum of the K slices (in slice order), bias, optional residual; four columns
// per thread.
__global__ void __launch_bounds__(256)
linear_finish_kernel(LinearArgs p, int slices) {
  const int quads_per_row = p.N / 4;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= p.M * quads_per_row) return;
  const int row = idx / quads_per_row, col = 4 * (idx - row * quads_per_row);
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = 0; s < slices; ++s) {
    const f32x4 part = *reinterpret_cast<const f32x4*>(
        p.partial + ((size_t)s * p.M + row) * p.N + col);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += part[i];
  }
  if (p.bias) {
    float b[4];
    unpack4(*reinterpret_cast<const u32x2*>(
                reinterpret_cast<const uint16_t*>(p.bias) + col), b);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += b[i];
  }
  const size_t at = out_index(row, col, p.M, p.group_width);
  if (p.residual) {
    float res[4];
    unpack4(*reinterpret_cast<const u32x2*>(
                reinterpret_cast<const uint16_t*>(p.residual) + at), res);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = round_to_bf16(v[i]) + res[i];
  }
  const u32x2 ov = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(p.out) + at) = ov;
}

// One 16-byte item of the packed matrix per thread.  Source layouts:
//   0: [N, K] (torch.nn.Linear.weight)
//   1: [G, K, N / G] (the reference's Einsum weight "cdD", layers.py:97-101;
//      weight row n = g (N / G) + j is w[g, :, j])
// pair: tile 2 b is rows 32 b .. of the first half of the rows, tile 2 b + 1
// the same rows of the second half.
__global__ void __launch_bounds__(256)
linear_pack_kernel(const uint16_t* __restrict__ w, u32x4* __restrict__ packed,
                   int N, int K, int layout, int groups, int pair) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int ksteps = K / 16;
  if (idx >= (int64_t)(N / 32) * ksteps * 64) return;
  const int lane = (int)(idx & 63);
  const int ks = (int)((idx >> 6) % ksteps);
  const int tile = (int)((idx >> 6) / ksteps);
  int row = tile * 32 + (lane & 31);
  if (pair) row = (tile & 1) * (N / 2) + (tile >> 1) * 32 + (lane & 31);
  const int k = ks * 16 + 8 * (lane >> 5);
  u32x4 v;
  if (layout == 0) {
    v = *reinterpret_cast<const u32x4*>(w + (size_t)row * K + k);
  } else {
    const int gw = N / groups;
    const int grp = row / gw, j = row - grp * gw;
    const uint16_t* src = w + ((size_t)grp * K + k) * gw + j;
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = src[(size_t)i * gw];
    v = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16),
              e[6] | (e[7] << 16)};
  }
  packed[idx] = v;
}

template <int NT, int MODE, int XR, bool BESIDE, bool HALF>
hipError_t launch_rows_of(const LinearArgs& a, dim3 grid, hipStream_t s) {
  constexpr int lds = kWaves * wave_lds_bytes(NT, XR > 32 ? 2 : 1);
  static OncePerDevice once;  // one per instantiation of this launcher
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)linear_rows_kernel<NT, MODE, XR, BESIDE, HALF>, lds);
  if (e != hipSuccess) return e;
  linear_rows_kernel<NT, MODE, XR, BESIDE, HALF><<<grid, kWaves * 64, lds, s>>>(a);
  return hipGetLastError();
}

// How many rows of x a launch loads and stages.  us a layer, replayed from a
// graph over 16 sets of weights, always 64 rows and without the barrier that
// keeps the next chunk's loads in front of the products / as it is:
//   rows                     1           16           32           64
//   K 2560, N 2560     8.7 /  6.5   8.7 /  7.6   9.9 /  9.1  11.8 / 11.3
//   K 2560, N 5120    10.6 /  7.6  10.8 /  9.3  10.3 / 10.1  12.6 / 12.1
//   K 7680, N 2560    12.7 / 11.2  13.1 / 12.0  14.6 / 13.6  17.1 / 16.2
//   K 4096, N 8192    17.8 / 14.5  17.9 / 14.4  17.9 / 15.4  20.7 / 18.5
// (8 staged rows are within 2 % of 16.  Fewer rows without the barrier are
// slower than 64, 10.0 us for one row at 2560 x 2560: the compiler moves the
// loads behind the products.)
template <int NT, int MODE, bool BESIDE = false, bool HALF = false>
hipError_t launch_rows(const LinearArgs& a, dim3 grid, hipStream_t s) {
  if (a.M <= 16) return launch_rows_of<NT, MODE, 16, BESIDE, HALF>(a, grid, s);
  if (a.M <= 32) return launch_rows_of<NT, MODE, 32, BESIDE, HALF>(a, grid, s);
  return launch_rows_of<NT, MODE, 64, BESIDE, HALF>(a, grid, s);
}

// two tiles per workgroup once that still leaves a workgroup for most CUs
bool two_tiles(int tiles) { return tiles % 2 == 0 && tiles / 2 >= 200; }
// Half a tile while there is a CU for each: what a workgroup draws is what bounds it.  us a
// layer, replayed from a graph over 16 sets of weights, whole / half tiles:
//   rows                     1           16           32           64
//   K 2560, N 2560     6.0 /  5.5   7.1 /  6.1   8.4 /  7.4  10.6 /  9.8
//   K 2560, N 4096     6.4 /  5.9   7.4 /  6.4   8.8 /  7.8  11.0 / 10.3
//   K 4096, N 4096     9.6 /  8.5   9.9 /  8.5  11.5 / 10.1  14.6 / 13.6
//   K 1024, N 2048     4.1 /  3.8   4.2 /  3.9   4.7 /  4.3   5.8 /  5.6
// Of short rows a workgroup is mostly what it begins and ends with, and more than a few of
// them are better read once for a whole tile (whole over half; 2.3 to 4 us a layer):
//   rows                  1     4    16    32
//   K 128, N 1024      1.06  1.04  0.98  0.97
//   K 128, N 4096      1.00  1.00  0.92  0.92
//   K 256, N 2048      1.02  1.04  0.99  0.95
//   K 512, N 2048      1.09  1.09  1.04  1.03
bool half_tiles(int tiles, int M, int K) {
  return 2 * tiles <= 256 && (K >= 512 || M <= 4);
}

template <int NT, int MODE, int XR, int CPW, bool BESIDE>
hipError_t launch_normed_of(const NormedLinearArgs& a, int blocks, hipStream_t s) {
  constexpr int lds = kWaves * wave_lds_bytes(NT, XR > 32 ? 2 : 1);
  static OncePerDevice once;
  const auto kernel = linear_rows_normed_kernel<NT, MODE, XR, CPW, BESIDE>;
  hipError_t e = set_max_dynamic_lds(once, (const void*)kernel, lds);
  if (e != hipSuccess) return e;
  kernel<<<dim3((unsigned)(a.layer.M + blocks + (BESIDE ? kCopiers : 0))), kWaves * 64,
           lds, s>>>(a);
  return hipGetLastError();
}
constexpr int kNormedChunks = 5;  // of a wave: K 2560
template <int NT, int MODE, bool BESIDE>
hipError_t launch_normed_rows(const NormedLinearArgs& a, int blocks, hipStream_t s) {
  constexpr int CPW = kNormedChunks;
  if (a.layer.M <= 16) return launch_normed_of<NT, MODE, 16, CPW, BESIDE>(a, blocks, s);
  if (NT == 2 || a.layer.M <= 32)
    return launch_normed_of<NT, MODE, 32, CPW, BESIDE>(a, blocks, s);
  // (pairs end at 32 rows: linear_rows_normed_serve)
  return launch_normed_of<1, MODE == kGeluPair ? kStore : MODE, 64, CPW, BESIDE>(a, blocks, s);
}

}  // namespace

// How many slices of K the grid takes: more than one only where the weight
// rows alone leave most CUs idle and K is long enough to share out.
int linear_rows_k_slices(int K, int N) {
  const int tiles = N / 32;
  if (tiles <= 96 && K >= 5120) return 3;
  return 1;
}

hipError_t launch_linear_pack(const void* w, void* packed, int N, int K,
                              int layout, int groups, int pair, hipStream_t s) {
  const int64_t items = (int64_t)(N / 32) * (K / 16) * 64;
  linear_pack_kernel<<<dim3((unsigned)((items + 255) / 256)), 256, 0, s>>>(
      (const uint16_t*)w, (u32x4*)packed, N, K, layout, groups, pair);
  return hipGetLastError();
}

hipError_t launch_linear_rows_partial(const LinearArgs& a, int slices,
                                      hipStream_t s) {
  return launch_rows<1, kPartial>(a, dim3(a.N / 32, slices), s);
}

hipError_t launch_linear_rows(const LinearArgs& a, int gelu_pair,
                              hipStream_t s) {
  const int tiles = a.N / 32;
  if (gelu_pair)
    return launch_rows<2, kGeluPair>(a, dim3(tiles / 2, 1), s);
  const int slices = linear_rows_k_slices(a.K, a.N);
  if (slices > 1) {
    hipError_t e = launch_rows<1, kPartial>(a, dim3(tiles, slices), s);
    if (e != hipSuccess) return e;
    const int quads = a.M * (a.N / 4);
    linear_finish_kernel<<<dim3((quads + 255) / 256), 256, 0, s>>>(a, slices);
    return hipGetLastError();
  }
  if (two_tiles(tiles)) return launch_rows<2, kStore>(a, dim3(tiles / 2, 1), s);
  if (half_tiles(tiles, a.M, a.K))
    return launch_rows<1, kStore, false, true>(a, dim3(2 * tiles, 1), s);
  return launch_rows<1, kStore>(a, dim3(tiles, 1), s);
}

// A layer whose K is not split (the caller has seen to it), and the copy beside it:
// 160 workgroups at N 5120 leave the CUs that do it idle otherwise.
hipError_t launch_linear_rows_beside(const LinearArgs& a, hipStream_t s) {
  const int tiles = a.N / 32;
  if (two_tiles(tiles))
    return launch_rows<2, kStore, true>(a, dim3(tiles / 2 + kCopiers, 1), s);
  return launch_rows<1, kStore, true>(a, dim3(tiles + kCopiers, 1), s);
}

// Whether a layer (or layers packed together) with the norm in front of it is one launch:
// K as the kernel is made for (a wave's weights fill its registers), single tiles, pairs
// for up to 32 rows (us, two launches / one: N 5120 at 40, 64 rows 14.2 / 12.5, 16.2 /
// 13.5, N 3072 14.1 / 12.1, 15.7 / 13.4; pairs of N 15360 21.6 / 22.0, 23.1 / 23.1: the
// workgroups are more than the CUs).
bool linear_rows_normed_serve(int M, int K, int N, int gelu_pair) {
  return M > 0 && M <= (gelu_pair ? 32 : kNormFlags) &&
         K == kNormedChunks * kWaves * 64 && N % 32 == 0 &&
         (gelu_pair || !two_tiles(N / 32));
}

hipError_t launch_linear_rows_normed(const NormedLinearArgs& a, int gelu_pair,
                                     hipStream_t s) {
  const int tiles = a.layer.N / 32;
  if (gelu_pair) return launch_normed_rows<2, kGeluPair, false>(a, tiles / 2, s);
  return a.layer.copy_items ? launch_normed_rows<1, kStore, true>(a, tiles, s)
                            : launch_normed_rows<1, kStore, false>(a, tiles, s);
}

}  // namespace rg
