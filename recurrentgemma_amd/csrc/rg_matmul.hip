// Linear layers of many rows in bf16 (the nn.Linear and stacked layers of
// recurrentgemma/torch/modules.py:605-760 and :404-476 on prompts and training
// batches): C[m, n] = sum_k of an M-side times an N-side operand, float32 sums, one
// rounding.  Each side comes with the contraction as its contiguous dimension
// (activations [rows, features], weights [out, in]) or as its slow one (weights
// [in, out]; both sides of a weight gradient), so the three directions of a layer are
// one kernel:
//   kMatmulForward   x [M, K] . w [N, K]^T (+ bias)
//   kMatmulBack      dy [M, K] . w [K, N], the contraction in one stretch or two
//                    (two layers that share an input: one product over both)
//   kMatmulWeights   dy [K, M]^T . x [K, N]
//   kMatmulGeluPair  gelu(x . w [K, N] + bias) * (x . w2 [K, N] + bias2)
// Up to kMaxMatmuls products go out as one launch, tile after tile.
//
// One workgroup of four waves, one per SIMD, per tile of 32 MB x 64 NB outputs (256 x
// 320 for a large product).  Both operands go global -> LDS by the memory pipe in steps
// of 64 along the contraction, two stages; a wave multiplies a quarter of the tile from
// LDS with v_mfma_f32_16x16x32_bf16, operand fragments of the next half step on their
// way while those of this one are multiplied.  A side whose contraction is the slow
// dimension is staged as it lies and read with ds_read_b64_tr_b16, which hands out
// columns.
//
// What bounds it is power: the matrix pipe is busy 82-86 % of the main loop's cycles
// and the clock gives way to 1.6-1.85 GHz under it (with zeros for operands the same
// loop runs at 2.25).  So what costs energy decides:
//  - 16x16x32 instructions instead of 32x32x16 (half the accumulator traffic for the
//    same product; 1.40-1.55 GHz at 94 % busy): 8192 x 5120 x 2560 168 -> 156 us.
//  - Tiles 320 wide: fewer LDS reads per product than 256 x 256, and the widths that
//    are multiples of 320 come out even on 256 CUs (8192 x 2560: 256 tiles for 320).
//  - 16-byte chunks of an LDS row permuted by the row's number, so that operand reads
//    meet no bank twice; full 128-byte lines per row in every load.
// A stage's lines are asked into L2 one step before the stage is loaded (each
// workgroup its share of the panels that the workgroups of its XCD read together): a
// stage has one step to arrive, which a miss in L2 does not make (8192 x 5120 x 2560
// 176 -> 168 us).
// Rates in TFLOP/s, operands in memory, against the library's: rows 8192, 5120 x 2560
// forward 1370 (870); back through two 2560 x 2560 layers 1370 (930); three weight
// gradients of 2560 x 2560 over 8192 rows 1340 (770).
#include <math.h>

#include "rg_common.h"
#include "rg_internal.h"
#include "rg_matrix_asm.h"

namespace rg {
namespace {

using namespace matrix_asm;

constexpr int kStep = 64;           // of the contraction, per stage
constexpr int kPanelBytes = 8192;   // 64 x 64 values of one operand
constexpr int kAccBlocks = 64;      // 16 x 16 results in a[0:255], the rest in VGPRs

// Which tile a workgroup has: contiguous runs of tiles per XCD (workgroups go to the
// eight XCDs in turn); inside a product eight tile rows side by side, so that the 32
// workgroups of an XCD read eight panels of rows and four of columns between them.
struct TileAt {
  int which, tm, tn;
};
__device__ __forceinline__ TileAt tile_at(const MatmulArgs& args, int tile_m, int tile_n) {
  unsigned id = blockIdx.x;
  const unsigned per_xcd = gridDim.x / 8;
  if (id < 8 * per_xcd) id = (id & 7) * per_xcd + (id >> 3);
  int which = 0;
  while (which + 1 < args.count && (int)id >= args.p[which + 1].first_tile) ++which;
  const MatmulProblem& p = args.p[which];
  id -= p.first_tile;
  const int tiles_n = (p.N + tile_n - 1) / tile_n, tiles_m = (p.M + tile_m - 1) / tile_m;
  const int group = (int)id / (8 * tiles_n), in_group = (int)id % (8 * tiles_n);
  const int group_m = tiles_m - 8 * group < 8 ? tiles_m - 8 * group : 8;
  return {which, 8 * group + in_group % group_m, in_group / group_m};
}

// The descriptor of an operand from a tile's first row (slow: column) to its end.
__device__ __forceinline__ u32x4 operand(const MatmulProblem& p, const void* base, bool slow,
                                         int first, int rows, int ld) {
  const int64_t skip = slow ? 2ll * first : 2ll * first * ld;
  const int64_t all =
      slow ? 2 * ((int64_t)(p.K - 1) * ld + rows) : 2 * ((int64_t)(rows - 1) * ld + p.K);
  return scalar_rsrc((const char*)base + skip, all - skip);
}

// A load instruction fills 1 KB: eight rows of a panel (rows of the operand, or of
// the contraction where that is the slow dimension), 128 bytes each, their 16-byte
// chunks permuted by the row's number.
__device__ __forceinline__ uint32_t load_offset(int lane, bool slow, int ld2) {
  const int lr = lane >> 3, lc = lane & 7;
  return (uint32_t)(lr * ld2 + 16 * (slow ? lc ^ ((lr & 3) << 1) : lc ^ lr));
}

// Operand fragments: lane (n = lane % 16, quarter = lane / 16) holds row n of a 16-row
// block, contraction indices 8 quarter .. + 7 of a half step.  Addresses per half step,
// or (slow) per block of a panel, of rows 8 quarter + n / 4 and four on.
__device__ __forceinline__ void lane_address(int lane, bool slow, uint32_t base,
                                             uint32_t (&a)[4]) {
  const int n = lane & 15, quarter = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    a[i] = base + (slow ? (uint32_t)(128 * (8 * quarter + (n >> 2)) +
                                     16 * ((2 * i + ((n & 3) >> 1)) ^ ((n >> 2) << 1)) +
                                     8 * (n & 1))
                        : (uint32_t)(128 * n + 16 * ((4 * i + quarter) ^ (n & 7))));
}
__device__ __forceinline__ f32x4 fragment(bool slow, const uint32_t (&a)[4], uint32_t stage,
                                          int block, int panel, int half_step) {
  if (!slow)
    return *reinterpret_cast<const lds_f32x4*>((lds_byte*)(uintptr_t)(a[half_step] + stage) +
                                               2048 * block);
  union {
    s16x4 h[2];
    f32x4 v;
  } u;
  lds_byte* const at = (lds_byte*)(uintptr_t)(a[block] + stage) + panel * kPanelBytes +
                       4096 * half_step;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 512));
  return u.v;
}

// A wave's results, MB x BLOCKS blocks of 16 x 16, to C: lane (n, quarter) has row n of a
// block of 16 rows, columns 4 quarter .. + 3 of one of 16 columns.  row0: the wave's
// first row behind m0; column(nb): the first column of block nb (and the next: nb is
// even).  PAIR: the second half of the blocks are the second weight's.
template <bool PAIR, int MB, int BLOCKS, bool RUNS, class Value, class Column>
__device__ __forceinline__ void store_tile(const MatmulArgs& args, const MatmulProblem& p,
                                           int m0, int row0, int lane, Value&& value,
                                           Column&& column) {
  const int n = lane & 15, quarter = lane >> 4;
  const int64_t skip = RUNS ? 0 : 2ll * m0 * p.ldc;
  const __amdgpu_buffer_rsrc_t rc = make_rsrc(
      (char*)p.c + skip,
      (uint32_t)(2 * ((int64_t)((RUNS ? args.rows : p.M) - 1) * p.ldc + p.N) - skip));
  // this lane's row of each block of 16
  uint32_t row_at[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    if (RUNS) {
      const int run = (m0 + row0) / 8 + 2 * mb + (n >> 3);
      row_at[mb] = 8 * run < p.M ? (uint32_t)(args.runs[run] + (n & 7)) * 2u * (uint32_t)p.ldc
                                 : kBufferOutOfRange;
    } else {
      row_at[mb] = (uint32_t)(row0 + n + 16 * mb) * 2u * (uint32_t)p.ldc;
    }
  }
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.bias, p.bias ? 2u * (uint32_t)p.N : 0u);
  const __amdgpu_buffer_rsrc_t rb2 =
      make_rsrc(p.bias2, PAIR && p.bias2 ? 2u * (uint32_t)p.N : 0u);
  struct Four {
    float v[4];
  };
  auto bias_at = [&](__amdgpu_buffer_rsrc_t r, int col) {
    const u32x2 b = __builtin_amdgcn_raw_buffer_load_b64(r, 2u * (uint32_t)col, 0, 0);
    return Four{{__uint_as_float(b[0] << 16), __uint_as_float(b[0] & 0xffff0000u),
                 __uint_as_float(b[1] << 16), __uint_as_float(b[1] & 0xffff0000u)}};
  };
  // two blocks of 16 columns side by side: a quarter trades one of its two runs of four
  // columns for its neighbour's and has eight in a row
  for_n<(PAIR ? BLOCKS / 2 : BLOCKS) / 2>([&](auto PB) {
    constexpr int nb = 2 * decltype(PB)::value;
    const int col = column(nb);
    Four bias[2], bias2[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      bias[e] = bias_at(rb, col + 16 * e + 4 * quarter);
      if (PAIR) bias2[e] = bias_at(rb2, col + 16 * e + 4 * quarter);
    }
    const int at = col + 16 * (quarter & 1) + 4 * (quarter & 2);
    for_n<MB>([&](auto MBI) {
      constexpr int mb = decltype(MBI)::value;
      uint32_t w[2][2];
      for_n<4>([&](auto ER) {
        constexpr int e = decltype(ER)::value / 2, r = 2 * (decltype(ER)::value % 2);
        auto two = [&](auto BLK, const Four& b) {
          return pack_bf16x2(value(BLK, std::integral_constant<int, r>{}) + b.v[r],
                             value(BLK, std::integral_constant<int, r + 1>{}) + b.v[r + 1]);
        };
        const uint32_t one = two(std::integral_constant<int, (nb + e) * MB + mb>{}, bias[e]);
        if constexpr (PAIR)
          w[e][r / 2] = gelu_mul_bf16x2(
              two(std::integral_constant<int, (BLOCKS / 2 + nb + e) * MB + mb>{}, bias2[e]),
              one);
        else
          w[e][r / 2] = one;
      });
      const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
      buffer_store_16(u32x4{s0[0], s1[0], s0[1], s1[1]}, rc,
                      at < p.N ? row_at[mb] + 2u * (uint32_t)at : kBufferOutOfRange, 0);
    });
  });
}

// KIND as in rg_internal.h; wave tile 16 MB x 32 NB.  RUNS: the rows of a tile are runs of
// eight wherever they lie (a load instruction has eight rows: a scalar offset each, made
// once), so that padding between sequences is neither read nor multiplied.
template <int KIND, int MB, int NB, bool RUNS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
matmul_bf16_kernel(MatmulArgs args) {
  constexpr bool kPair = KIND == kMatmulGeluPair;
  // sides whose contraction is the slow dimension
  constexpr bool kSlowM = KIND == kMatmulWeights;
  constexpr bool kSlowN = KIND != kMatmulForward;
  constexpr bool kTwoStretches = KIND == kMatmulBack;
  constexpr int kPanelsM = MB / 2, kPanelsN = NB;
  constexpr int kTileM = 32 * MB;
  constexpr int kTileN = kPair ? 32 * NB : 64 * NB;  // columns of C
  constexpr int kStage = (kPanelsM + kPanelsN) * kPanelBytes;
  constexpr int kLoads = 2 * (kPanelsM + kPanelsN);  // per wave and stage
  constexpr int kLoadsEarly = kLoads / 2;            // behind the barrier at once
  constexpr int kBlocksN = 2 * NB;                   // of 16, per wave
  constexpr int kMfmas = MB * kBlocksN;              // per half step and wave
  constexpr int kReads = MB + kBlocksN;
  extern __shared__ __align__(16) unsigned char matmul_lds[];
  lds_byte* const lds = (lds_byte*)matmul_lds;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;

  const TileAt at = tile_at(args, kTileM, kTileN);
  const MatmulProblem& p = args.p[at.which];
  const int tm = at.tm, tn = at.tn;
  const int m0 = tm * kTileM, n0 = tn * kTileN;
  const int ldm2 = 2 * p.ldm, ldn2 = 2 * p.ldn;  // bytes
  static_assert(!RUNS || (!kSlowM && !kTwoStretches), "");
  u32x4 rm = operand(p, p.m, kSlowM, RUNS ? 0 : m0, RUNS ? args.rows : p.M, p.ldm);
  u32x4 rn = operand(p, p.n, kSlowN, n0, p.N, p.ldn);
  u32x4 rn_up = rn;
  if (kPair) rn_up = operand(p, p.n2, kSlowN, n0, p.N, p.ldn);
  const int steps_one = (p.K + kStep - 1) / kStep;
  const int steps = kTwoStretches && p.m2 ? 2 * steps_one : steps_one;

  const uint32_t vm0 = load_offset(lane, kSlowM, ldm2), vn0 = load_offset(lane, kSlowN, ldn2);
  const uint32_t step_m = kSlowM ? kStep * ldm2 : 2 * kStep;
  const uint32_t step_n = kSlowN ? kStep * ldn2 : 2 * kStep;
  uint32_t vm = vm0, vn = vn0;
  // wave's part of panel i / 2: rows 32 (i % 2) + 8 wave .. + 7
  int scalar_offset[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = 32 * (i & 1) + 8 * wave;
    const bool is_m = i / 2 < kPanelsM;
    int panel = is_m ? i / 2 : i / 2 - kPanelsM;
    if (kPair && !is_m) panel %= NB / 2;
    scalar_offset[i] = (is_m ? kSlowM : kSlowN)
                           ? row * (is_m ? ldm2 : ldn2) + 128 * panel
                           : (64 * panel + row) * (is_m ? ldm2 : ldn2);
    // (behind the last run: the last once more, whose results are dropped)
    if (RUNS && is_m)
      scalar_offset[i] =
          args.runs[min((m0 + 64 * panel + row) / 8, p.M / 8 - 1)] * ldm2;
  }
  auto load = [&](uint32_t stage, auto I) {
    constexpr int i = decltype(I)::value;
    constexpr bool is_m = i / 2 < kPanelsM;
    constexpr bool is_up = kPair && i / 2 - kPanelsM >= NB / 2;
    const u32x4 r = is_m ? rm : is_up ? rn_up : rn;
    load_lds_16<i / 2 * kPanelBytes + (i & 1) * 4096>(
        stage + 1024 * (uint32_t)wave, is_m ? vm : vn, r, scalar_offset[i]);
  };

  // ---- lines of the step after a stage's, asked into L2 ------------------------------
  // wave 0: this workgroup's quarter of the M panels' lines, wave 1: its eighth of the
  // N panels'; what arrives goes to a corner of LDS that nobody reads.
  uint32_t vp0 = kBufferOutOfRange;
  if (wave == 0 && lane < 8 * MB) {
    constexpr int kLines = kTileM / 64;  // a row of the contraction is this many lines
    vp0 = kSlowM ? (uint32_t)((16 * (tn & 3) + lane / kLines) * ldm2 + 128 * (lane % kLines))
                 : (uint32_t)((8 * MB * (tn & 3) + lane) * ldm2);
    if (RUNS) {
      const int row = m0 + 8 * MB * (tn & 3) + lane;
      vp0 = (uint32_t)((args.runs[min(row / 8, p.M / 8 - 1)] + (row & 7)) * ldm2);
    }
  }
  if (wave == 1 && lane < 8 * NB) {
    constexpr int kLines = kTileN / 64;
    vp0 = kSlowN ? (uint32_t)((8 * (tm & 7) + lane % (8 * kLines) / kLines) * ldn2 +
                              128 * (lane % kLines))
                 : (uint32_t)((8 * NB * (tm & 7) + lane) * ldn2);
  }
  // (the pair's second weight is asked for by wave 2)
  if (kPair && wave == 2 && lane < 8 * NB)
    vp0 = (uint32_t)((8 * (tm & 7) + lane % (8 * (kTileN / 64)) / (kTileN / 64)) * ldn2 +
                     128 * (lane % (kTileN / 64)));
  u32x4 rp = wave == 0 ? rm : kPair && wave == 2 ? rn_up : rn;
  const uint32_t step_p = wave == 0 ? step_m : step_n;
  uint32_t vp = vp0 + step_p;
  auto prefetch = [&] {
    load_lds_4((uint32_t)(uintptr_t)lds + 2 * kStage + 256 * (uint32_t)wave, vp, rp);
  };
  int load_step = 0;
  auto advance = [&] {  // a stage's loads are out: on to the next step's
    ++load_step;
    vm += step_m;
    vn += step_n;
    vp += step_p;
    if (kTwoStretches && load_step == steps_one && steps > steps_one) {
      rm = operand(p, p.m2, kSlowM, m0, p.M, p.ldm);
      rn = operand(p, p.n2, kSlowN, n0, p.N, p.ldn);
      rp = wave == 0 ? rm : rn;
      vm = vm0;
      vn = vn0;
      vp = vp0 + step_p;
    }
    if (load_step >= steps) rm[2] = rn[2] = rn_up[2] = 0;  // nothing more is read
    if (load_step + 1 >= steps) rp[2] = 0;
  };

  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  uint32_t am[4], an[4];
  lane_address(lane, kSlowM, lds0 + wm * (MB / 4) * kPanelBytes, am);
  // The N side's blocks of a wave: 16 kBlocksN in a row, or (slow: whole panels are
  // wanted, for constant offsets) every second pair of blocks, or of each weight of a
  // pair the same panel.
  lane_address(lane, kSlowN,
               lds0 + kPanelsM * kPanelBytes +
                   (kPair ? wn * kPanelBytes : kSlowN ? 0 : wn * NB * 4096),
               an);
  if (kSlowN && !kPair && wn) {
    an[0] = an[2];
    an[1] = an[3];
  }
  f32x4 fm[2][MB], fn[2][kBlocksN];
  auto read = [&](uint32_t stage, int half_step, auto I) {
    constexpr int i = decltype(I)::value;
    if constexpr (i < MB) {
      fm[half_step][i] = kSlowM ? fragment(true, am, stage, i & 3, i >> 2, half_step)
                                : fragment(false, am, stage, i, 0, half_step);
    } else {
      constexpr int j = i - MB;
      fn[half_step][j] =
          kPair ? fragment(true, an, stage, j & 3, (j >> 2) * (NB / 2), half_step)
          : kSlowN ? fragment(true, an, stage, j & 1, j >> 1, half_step)
                   : fragment(false, an, stage, j, 0, half_step);
    }
  };

  // ---- main loop -----------------------------------------------------------------------
  constexpr int kInVgprs = MB * kBlocksN > kAccBlocks ? MB * kBlocksN - kAccBlocks : 0;
  f32x4 extra[kInVgprs > 0 ? kInVgprs : 1];
#pragma unroll
  for (int i = 0; i < kInVgprs; ++i) extra[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  take_accumulators();
  for_n<4 * (MB * kBlocksN - kInVgprs)>([&](auto I) { acc_zero<decltype(I)::value>(); });

  // a half step's matrix instructions, with what `between` issues behind each
  auto multiply = [&](auto HALF, auto&& between) {
    constexpr int half_step = decltype(HALF)::value;
    for_n<kMfmas>([&](auto I) {
      constexpr int i = decltype(I)::value, nb = i / MB, mb = i % MB;
      const f32x4 &a = fn[half_step][nb], &b = fm[half_step][mb];
      if constexpr (i < kAccBlocks) {
        acc_mfma<i>(a, b);
      } else {
        f32x4& c = extra[i - kAccBlocks];
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
      }
      __builtin_amdgcn_sched_barrier(0);
      between(I);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  constexpr int kReadEvery = kMfmas / kReads > 2 ? kMfmas / kReads - 1 : 2;
  constexpr int kEarlyEvery = kMfmas / kLoadsEarly;
  constexpr int kLateEvery = kMfmas / 20 > 2 ? kMfmas / 20 : 2;
  static_assert(kReadEvery * (kReads - 1) < kMfmas, "reads of a half step");
  static_assert(kLateEvery * (kLoads - kLoadsEarly) + 1 < kMfmas, "loads of a half step");
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;

  for_n<kLoads>([&](auto I) { load(lds0, I); });
  advance();
  for_n<kLoadsEarly>([&](auto I) { load(lds0 + kStage, I); });
  asm volatile("s_waitcnt vmcnt(%c0)\n\ts_barrier" ::"n"(kLoadsEarly) : "memory");
  for_n<kReads>([&](auto I) { read(0, 0, I); });
  uint32_t stage = 0;
  for (int step = 0; step < steps; ++step) {
    // First half step: this stage's second half is read, the next stage's loads end.
    const uint32_t next = kStage - stage;
    multiply(Zero{}, [&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (i % kReadEvery == 0 && i / kReadEvery < kReads)
        read(stage, 1, std::integral_constant<int, i / kReadEvery>{});
      if constexpr (i % kLateEvery == 1 && kLoadsEarly + i / kLateEvery < kLoads)
        load(lds0 + next, std::integral_constant<int, kLoadsEarly + i / kLateEvery>{});
      if constexpr (i == kLateEvery * (kLoads - kLoadsEarly) + 1) prefetch();
    });
    advance();
    // This wave has read all of this stage and its share of the next one is there
    // (everything but the prefetch): behind the barrier that holds for all four.
    asm volatile("s_waitcnt vmcnt(1) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    multiply(One{}, [&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (i % kReadEvery == 0 && i / kReadEvery < kReads)
        read(next, 0, std::integral_constant<int, i / kReadEvery>{});
      if constexpr (i % kEarlyEvery == 1 && i / kEarlyEvery < kLoadsEarly)
        load(lds0 + stage, std::integral_constant<int, i / kEarlyEvery>{});
    });
    stage = next;
  }
  // (no load outlives the workgroup's LDS; the last ones were out of range)
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < kInVgprs; ++i) asm volatile("" : "+v"(extra[i]));

  auto value = [&](auto BLK, auto R) -> float {
    constexpr int b = decltype(BLK)::value, r = decltype(R)::value;
    if constexpr (b < kAccBlocks) return acc_read<4 * b + r>();
    else return extra[b - kAccBlocks][r];
  };
  store_tile<kPair, MB, kBlocksN, RUNS>(args, p, m0, 16 * MB * wm, lane, value, [&](int nb) {
    return n0 + (kPair ? 64 * wn + 16 * nb
                 : kSlowN ? 32 * (nb + wn)
                          : 32 * NB * wn + 16 * nb);
  });
}

// The same for few rows, whose large tiles would leave most CUs idle: tiles of 64 x 64 or
// 128 x 128 (64 x 128 of a pair's columns twice), which several stages of loads on their
// way keep going: a step is short against the way of its operands from memory.  Wave tile
// 16 MB x 16 NB.
template <int KIND, int MB, int NB, int STAGES>
__global__ void __launch_bounds__(256) matmul_small_bf16_kernel(MatmulArgs args) {
  constexpr bool kPair = KIND == kMatmulGeluPair;
  constexpr bool kSlowM = KIND == kMatmulWeights;
  constexpr bool kSlowN = KIND != kMatmulForward;
  constexpr bool kTwoStretches = KIND == kMatmulBack;
  static_assert(!kPair || NB == 4, "a panel of each weight");
  constexpr int kPanelsM = MB / 2, kPanelsN = NB / 2;
  constexpr int kTileM = 32 * MB, kTileN = kPair ? 16 * NB : 32 * NB;
  constexpr int kStage = (kPanelsM + kPanelsN) * kPanelBytes;
  constexpr int kLoads = 2 * (kPanelsM + kPanelsN);  // per wave and stage
  extern __shared__ __align__(16) unsigned char matmul_lds[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte*)matmul_lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const TileAt at = tile_at(args, kTileM, kTileN);
  const MatmulProblem& p = args.p[at.which];
  const int m0 = at.tm * kTileM, n0 = at.tn * kTileN;
  const int ldm2 = 2 * p.ldm, ldn2 = 2 * p.ldn;  // bytes
  u32x4 rm = operand(p, p.m, kSlowM, m0, p.M, p.ldm);
  u32x4 rn = operand(p, p.n, kSlowN, n0, p.N, p.ldn);
  u32x4 rn_up = rn;
  if (kPair) rn_up = operand(p, p.n2, kSlowN, n0, p.N, p.ldn);
  const int steps_one = (p.K + kStep - 1) / kStep;
  const int steps = kTwoStretches && p.m2 ? 2 * steps_one : steps_one;
  const uint32_t vm0 = load_offset(lane, kSlowM, ldm2), vn0 = load_offset(lane, kSlowN, ldn2);
  const uint32_t step_m = kSlowM ? kStep * ldm2 : 2 * kStep;
  const uint32_t step_n = kSlowN ? kStep * ldn2 : 2 * kStep;
  uint32_t vm = vm0, vn = vn0;
  int load_step = 0;
  uint32_t load_stage = lds0 + 1024 * (uint32_t)wave;
  const uint32_t stages_end = load_stage + STAGES * kStage;
  auto load_next = [&] {  // the next step's operands into the next stage
    for_n<kLoads>([&](auto I) {
      constexpr int i = decltype(I)::value;
      constexpr bool is_m = i / 2 < kPanelsM;
      constexpr bool is_up = kPair && i / 2 - kPanelsM >= kPanelsN / 2;
      constexpr int panel = is_m ? i / 2 : kPair ? 0 : i / 2 - kPanelsM;
      const int row = 32 * (i & 1) + 8 * wave;
      const int ld2 = is_m ? ldm2 : ldn2;
      const int where = (is_m ? kSlowM : kSlowN) ? row * ld2 + 128 * panel
                                                 : (64 * panel + row) * ld2;
      const u32x4 r = is_m ? rm : is_up ? rn_up : rn;
      load_lds_16<i / 2 * kPanelBytes + (i & 1) * 4096>(load_stage, is_m ? vm : vn, r, where);
    });
    load_stage += kStage;
    if (load_stage == stages_end) load_stage -= STAGES * kStage;
    ++load_step;
    vm += step_m;
    vn += step_n;
    if (kTwoStretches && load_step == steps_one && steps > steps_one) {
      rm = operand(p, p.m2, kSlowM, m0, p.M, p.ldm);
      rn = operand(p, p.n2, kSlowN, n0, p.N, p.ldn);
      vm = vm0;
      vn = vn0;
    }
    if (load_step >= steps) rm[2] = rn[2] = rn_up[2] = 0;  // nothing more is read
  };

  // A wave's blocks: 16 MB rows and 16 NB columns in a row (slow sides: blocks of a panel,
  // of two waves where it takes half of one; a pair: the same half of either weight's).
  uint32_t am[4], an[4];
  lane_address(lane, kSlowM, lds0 + wm * MB * 2048, am);
  lane_address(lane, kSlowN, lds0 + kPanelsM * kPanelBytes + (kPair ? 0 : wn * NB * 2048), an);
  auto half_panels = [&](uint32_t (&a)[4], int w) {  // (w * 4096 went into the base)
    if (!w) return;
    a[0] = a[2] - 4096;
    a[1] = a[3] - 4096;
  };
  if (kSlowM && MB == 2) half_panels(am, wm);
  if (kSlowN && NB == 2) half_panels(an, wn);
  if (kPair && wn) {
    an[0] = an[2];
    an[1] = an[3];
  }
  f32x4 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < MB * NB; ++i) acc[i / MB][i % MB] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for_n<STAGES - 1>([&](auto) { load_next(); });
  uint32_t stage = 0;
  int step = 0;
  do {
    // This step's operands are there, and everyone has read the last step's.
    asm volatile("s_waitcnt vmcnt(%c0)\n\ts_barrier" ::"n"((STAGES - 2) * kLoads) : "memory");
    load_next();
    f32x4 fm[2][MB], fn[2][NB];
    for_n<2>([&](auto H) {
      constexpr int h = decltype(H)::value;
      for_n<MB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        fm[h][i] = fragment(kSlowM, am, stage, i, 0, h);
      });
      for_n<NB>([&](auto J) {
        constexpr int j = decltype(J)::value;
        fn[h][j] = kPair ? fragment(true, an, stage, j & 1, j >> 1, h)
                         : fragment(kSlowN, an, stage, j, 0, h);
      });
    });
    for_n<2 * MB * NB>([&](auto I) {
      constexpr int i = decltype(I)::value, h = i / (MB * NB), nb = i / MB % NB, mb = i % MB;
      const f32x4 &a = fn[h][nb], &b = fm[h][mb];
      f32x4& c = acc[nb][mb];
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
    });
    stage = stage + kStage == STAGES * kStage ? 0 : stage + kStage;
  } while (++step < steps);
  // (no load outlives the workgroup's LDS; the last ones were out of range)
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < MB * NB; ++i) asm volatile("" : "+v"(acc[i / MB][i % MB]));
  auto value = [&](auto BLK, auto R) -> float {
    constexpr int b = decltype(BLK)::value;
    return acc[b / MB][b % MB][decltype(R)::value];
  };
  store_tile<kPair, MB, NB, false>(args, p, m0, 16 * MB * wm, lane, value, [&](int nb) {
    return n0 + (kPair ? 32 * wn + 16 * nb : 16 * NB * wn + 16 * nb);
  });
}

constexpr int kCus = 256;

// Fills in each product's first tile; how many there are.
unsigned first_tiles(MatmulArgs& a, int rows, int cols) {
  int64_t tiles = 0;
  for (int i = 0; i < a.count; ++i) {
    a.p[i].first_tile = (int)tiles;
    tiles += (int64_t)((a.p[i].M + rows - 1) / rows) * ((a.p[i].N + cols - 1) / cols);
  }
  return (unsigned)tiles;
}

template <int KIND, int MB, int NB, bool RUNS = false>
hipError_t launch_tiles(MatmulArgs& a, hipStream_t s) {
  if constexpr (!RUNS && (KIND == kMatmulForward || KIND == kMatmulGeluPair))
    if (a.runs) return launch_tiles<KIND, MB, NB, true>(a, s);
  constexpr int kTileN = KIND == kMatmulGeluPair ? 32 * NB : 64 * NB;
  constexpr int kLds = 2 * (MB / 2 + NB) * kPanelBytes + 4 * 256;
  static OncePerDevice once;
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)matmul_bf16_kernel<KIND, MB, NB, RUNS>, kLds);
  if (e != hipSuccess) return e;
  matmul_bf16_kernel<KIND, MB, NB, RUNS><<<dim3(first_tiles(a, 32 * MB, kTileN)), 256, kLds, s>>>(a);
  return hipGetLastError();
}

template <int KIND, int MB, int NB, int STAGES>
hipError_t launch_small(MatmulArgs& a, hipStream_t s) {
  constexpr int kTileN = KIND == kMatmulGeluPair ? 16 * NB : 32 * NB;
  constexpr int kLds = STAGES * (MB / 2 + NB / 2) * kPanelBytes;
  static OncePerDevice once;
  const auto kernel = matmul_small_bf16_kernel<KIND, MB, NB, STAGES>;
  hipError_t e = set_max_dynamic_lds(once, (const void*)kernel, kLds);
  if (e != hipSuccess) return e;
  kernel<<<dim3(first_tiles(a, 32 * MB, kTileN)), 256, kLds, s>>>(a);
  return hipGetLastError();
}

template <int KIND>
hipError_t launch_kind(MatmulArgs& a, int tile, hipStream_t s) {
  if (tile == 5) return launch_small<KIND, 4, 4, 4>(a, s);
  if constexpr (KIND == kMatmulGeluPair) {
    if (tile == 4) return launch_small<KIND, 2, 4, 4>(a, s);
  } else {
    if (tile == 4) return launch_small<KIND, 2, 2, 5>(a, s);
  }
  if (tile == 0) return launch_tiles<KIND, 8, 4>(a, s);
  if (tile == 2) return launch_tiles<KIND, 4, 4>(a, s);
  if constexpr (KIND != kMatmulGeluPair) {
    if (tile == 1) return launch_tiles<KIND, 8, 5>(a, s);
    if (tile == 3) return launch_tiles<KIND, 4, 5>(a, s);
  }
  return hipErrorInvalidValue;
}

// What a launch takes with each tile, in microseconds: once, per round of the chip, and per
// step of the contraction in it.  (Large tiles measured at 8192 and 16000 rows of 2560 to
// 7680 and 8192 x 4096 x 4096, small ones at 70 to 3000 rows of 2560 to 7680: 64 x 64
// within 15 % at 2560, 100 rows 11, 300 rows 12, 600 rows 19, 2048 rows 41.)
struct Tile {
  int rows, cols;
  float step_us, round_us, once_us;
};
constexpr int kTileForms = 6;
constexpr Tile kTiles[kTileForms] = {{256, 256, 1.37f, 9.0f, 0.0f}, {256, 320, 1.78f, 10.0f, 0.0f},
                                     {128, 256, 0.80f, 7.0f, 0.0f}, {128, 320, 1.00f, 7.0f, 0.0f},
                                     {64, 64, 0.185f, 1.0f, 3.5f},  {128, 128, 0.53f, 1.0f, 3.0f}};
// (a pair's tiles have half the columns; the small ones, 64 x 64 and 128 x 64, once in a
// CU, stream two weights)
constexpr Tile kPairTiles[kTileForms] = {{256, 128, 1.37f, 9.0f, 0.0f}, {0, 0, 0, 0, 0},
                                         {128, 128, 0.80f, 7.0f, 0.0f}, {0, 0, 0, 0, 0},
                                         {64, 64, 0.38f, 2.0f, 3.0f},   {128, 64, 0.57f, 2.0f, 3.0f}};

int64_t tiles_of(const MatmulProblem& p, int rows, int cols) {
  return (int64_t)((p.M + rows - 1) / rows) * ((p.N + cols - 1) / cols);
}
int steps_of(const MatmulProblem& p, int kind) {
  const int one = (p.K + kStep - 1) / kStep;
  return kind == kMatmulBack && p.m2 ? 2 * one : one;
}
float rounds(int64_t tiles) { return (float)((tiles + kCus - 1) / kCus); }

// The tile with which a launch takes least, in whole rounds of the chip.
float best_tile(const MatmulArgs& a, int kind, int* tile) {
  float best = 0.0f;
  *tile = -1;
  for (int t = 0; t < kTileForms; ++t) {
    const Tile& form = kind == kMatmulGeluPair ? kPairTiles[t] : kTiles[t];
    if (!form.rows || (a.runs && t > 3)) continue;  // (runs: large tiles alone)
    int64_t tiles = 0;
    int steps = 0;
    for (int i = 0; i < a.count; ++i) {
      tiles += tiles_of(a.p[i], form.rows, form.cols);
      const int n = steps_of(a.p[i], kind);
      if (n > steps) steps = n;
    }
    const float us =
        form.once_us + rounds(tiles) * (form.round_us + steps * form.step_us);
    if (*tile < 0 || us < best) {
      best = us;
      *tile = t;
    }
  }
  return best;
}

bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

// What the kernel can address: 16-byte loads and stores, offsets below 2^31.
bool matmul_serves(const MatmulArgs& a, int kind) {
  if (a.count < 1 || a.count > kMaxMatmuls) return false;
  if (a.runs && (kind == kMatmulBack || kind == kMatmulWeights || a.rows < 8)) return false;
  for (int i = 0; i < a.count; ++i) {
    const MatmulProblem& p = a.p[i];
    if (p.M < 1 || p.N < 8 || p.K < 1 || p.N % 8) return false;
    if (kind == kMatmulWeights ? p.M % 8 : p.K % kStep) return false;
    if ((p.ldm | p.ldn | p.ldc) % 8) return false;
    if (a.runs && p.M % 8) return false;
    const int64_t rows_c = a.runs ? a.rows : p.M;
    const int64_t rows_m = kind == kMatmulWeights ? p.K : rows_c;
    const int64_t rows_n = kind == kMatmulForward ? p.N : p.K;
    // (a step past the end is asked for, and found out of range)
    if (rows_m >= (1 << 30) || rows_n >= (1 << 30) ||
        (rows_m + 512) * p.ldm >= (1ll << 30) || (rows_n + 512) * p.ldn >= (1ll << 30) ||
        (rows_c + 512) * p.ldc >= (1ll << 30))
      return false;
    for (const void* t : {p.m, p.n, p.m2, p.n2, p.bias, p.bias2, (const void*)p.c})
      if (!aligned(t)) return false;
    if (tiles_of(p, 64, 64) > (1 << 28)) return false;
  }
  return true;
}

// Whether a launch is ahead of the library's products, one by one (weight gradients: at
// rg_linear_weight_grads).  Their time: whole rounds of 256 x 256 tiles at 1.3 us a step,
// or (few tiles) some 1.25 PFLOP/s and the way along the contraction; with the weights
// [in, out] 1.35 and more beside.  Measured over 64 to 32768 rows, widths 64 to 7680
// (library / this, us): forward 8192 x 2560 x 2560 93 / 74, two of them 189 / 147, 16376
// rows 233 / 149, 2048 rows 33 / 38, two of them 65 / 48, 300 rows 13 / 12, three of them
// 37 / 27, 1000 rows 24 / 25, 8192 x 4096 x 4096 171 / 184 (its 256 x 256 tiles come out
// even); back 8192 x 2560 x 2560 109 / 74, through two layers 230 / 138, 300 rows 17 / 14,
// 1500 rows 56 / 57 through two; the pair with its join, 8192 rows, 2560 -> 7680 494 + 60 /
// 481.
// Never less than 14 us, which counts the host's time and is right where calls are made
// one by one: nn.Linear keeps it for 21, a call here for 14 (three layers: 62 / 22), with
// 70, 300 or 1000 rows alike.  From a graph no host time counts, and a single layer with
// a long contraction and few tiles is behind there: 70 rows 2560 -> 2560 8.7 / 11.4 (100
// rows 10.8 / 11.3), 70 to 300 rows 2560 -> 256 7 / 11 and back 8 / 13.5, the pair so 17 /
// 19; of the other calls of a block 70 rows 2560 -> 2560 twice 17 / 12, thrice 30 / 13, the
// pair 2560 -> 7680 34 / 20, so that a captured step of more than 64 sequences gains.
static float library_us(const MatmulArgs& a, int kind) {
  constexpr float kCall = 14.0f;
  float library = 0.0f;
  for (int i = 0; i < a.count; ++i) {
    const MatmulProblem& p = a.p[i];
    const float gflop = 2e-9f * (float)p.M * (float)p.N * (float)p.K;
    const int steps = (p.K + kStep - 1) / kStep;
    if (kind == kMatmulForward) {
      const float whole = rounds(tiles_of(p, 256, 256)) * (6.0f + 1.3f * steps);
      const float few = 5.0f + 0.1f * steps + gflop / 1.25f;
      library += fmaxf(kCall, fminf(whole, few));
    } else {
      const bool two = kind == kMatmulGeluPair || p.n2;
      library += (two ? 2.0f : 1.0f) *
                 fmaxf(kCall, 6.0f + 0.13f * steps + gflop / 1.35f);
      if (kind == kMatmulGeluPair) library += 3.0f + 1.2e-6f * (float)p.M * (float)p.N;
    }
  }
  return library;
}

bool matmul_pays(const MatmulArgs& a, int kind) {
  int tile;
  return matmul_serves(a, kind) && best_tile(a, kind, &tile) < library_us(a, kind);
}

// What the products take where they are run better: here or by the library, which has
// no runs.
float matmul_us(const MatmulArgs& a, int kind) {
  int tile;
  const float own = matmul_serves(a, kind) ? best_tile(a, kind, &tile) : 1e30f;
  return a.runs ? own : fminf(own, library_us(a, kind));
}

hipError_t launch_matmul(MatmulArgs a, int kind, hipStream_t s) {
  if (!matmul_serves(a, kind)) return hipErrorInvalidValue;
  int tile;
  best_tile(a, kind, &tile);
  if (kind == kMatmulForward) return launch_kind<kMatmulForward>(a, tile, s);
  if (kind == kMatmulBack) return launch_kind<kMatmulBack>(a, tile, s);
  if (kind == kMatmulWeights) return launch_kind<kMatmulWeights>(a, tile, s);
  if (kind == kMatmulGeluPair) return launch_kind<kMatmulGeluPair>(a, tile, s);
  return hipErrorInvalidValue;
}

}  // namespace rg
