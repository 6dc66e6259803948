// The matrix products of RGLRU's gates in float32 (256-wide heads,
// recurrentgemma/torch/layers.py:127-137, called twice on the same x at
// :338-339), forwards and both ways backwards, on the bf16 matrix instructions:
//   forward   y_g[m, h, j] = sum_i x[m, h, i] w_g[h, i, j]
//   data      dx[m, h, i] += sum_g sum_j dy_g[m, h, j] w_g[h, i, j]
//   weights   dw_g[h, i, j] = sum_m x[m, h, i] dy_g[m, h, j]
//
// Every operand is cut into three bf16 pieces, each the nearest bf16 to what the
// pieces before it leave (v = hi + mid + lo: three times eight bits, all of a
// float32), and a product is the six products of pieces that weigh 2^-16 or more: what
// is left out, mid lo, lo mid and lo lo, is below 2^-26 of it.  v_mfma_f32_32x32x16_bf16 multiplies
// exactly and adds in float32; hi hi has an accumulator of its own, the five
// others share one whose roundings are 2^-8 times smaller, so a chain of K / 16
// roundings counts where the float32 instruction (32x32x2) has K / 2.  Six of
// them take 192 cycles for what eight of the others need 512, and vector
// instructions issue beside them.
//
// A piece has float32's range of exponents, so the last one of a value below 2^-110 =
// 8e-34 is no normal number any more and, further down, loses its digits.  Gradients
// (and x, where it meets them) are therefore cut 2^24 times as large, which makes every
// piece of every normal float32 a normal number or zero, and the results are scaled
// back, both exactly: dx of gradients of 1e-35 was off by 6e-6 of its norm and is as
// good as others now.  x and weights in the forward products and weights behind
// gradients are cut as they are: what they would gain lies 1e-34 below the bias, or the
// other share of dx, that it is added to.  (These scaled as well: float32 prefill of 8 x
// 2048 tokens, 2560 wide, 532 -> 539 us; as it is the kernels take what they took.)
//
// A workgroup of four waves owns 128 x 128 results, a wave 64 x 64 of them (two
// accumulators for each: half of its registers).  A stage is 16 k: its 2 x 128 x
// 16 floats are requested two stages ahead, cut between the matrix instructions
// of the stage before it and laid into the other of two LDS buffers in operand
// order; 48 KB, two workgroups a CU.  (Stages of 32 k cut between barriers, one
// buffer: 3 to 10 % slower.)  An operand whose memory runs along k is fetched
// eight k a lane with 16-byte loads, one whose memory runs along the result's rows
// or columns with eight loads of a row of lanes each: either way a lane has eight
// k of a row, and nothing is transposed.  Few rows: a quarter of the results and
// twice the k per stage (launch_rows).
//
// Bound by the matrix pipe at the clock that its power allows: 8192 rows of 10
// heads are 1.06 PFLOP/s of bf16 products, what large library products reach
// here.  us (and error of the result against 64 bits) / the float32 instruction's
// kernels that were here before (data: the library's two batched products):
//   rows               512         1001        2048        3003        8192
//   10 heads forward  17 /  20    24 /  34    37 /  51    49 /  65   122 / 162
//            data     25 /  39    26 /  57    41 /  94    48 /  83   120 / 195
//            weights  26 /  26    29 /  35    41 /  53    54 /  73   127 / 190
//   16 heads forward  20 /  22    27 /  36    50 /  67    72 /  97   210 / 267
//            data     25 /  38    29 /  46    50 /  84    75 / 152   210 / 330
//            weights  26 /  30    35 /  43    57 /  74    78 / 110   201 / 270
// (alone, operands in the caches; in the trace of a training step at 3003 rows 49, 51
// and 49 + 7)
// errors: forward 8.9e-8 / 2.1e-7, data 1.1e-7 / 2.4e-7, weights 7.7e-8 / 1.3e-7
// at 512 rows and 2.2e-7 / 4.7e-7 at 8192.
//
// Infinities and NaN: a piece of an infinity is no number, and scaled operands (from
// 2^104 = 2e31 on) or products of pieces (scaled: from 2^80 = 1e24 on) may overflow
// where the product does not.  Either leaves something that is not finite among a wave's results; such a wave computes them again with the
// float32 instruction and takes those for what was not finite (the others keep
// their bits whatever their neighbours hold).
#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kBW = 256;              // head width
constexpr int kThreads = 256;

// The two sizes of a workgroup: a wave has BLOCKS x BLOCKS blocks of 32 x 32
// results, a stage is as many k as give every thread eight of each operand.
template <int BLOCKS>
struct Size {
  static constexpr int tile = 64 * BLOCKS;    // results, each way
  static constexpr int stage = 32 / BLOCKS;   // k
  static constexpr int row = 2 * stage;       // bytes of an LDS row
  static constexpr int piece = tile * row;
  static constexpr int operand = 3 * piece;
  static constexpr int buffer = 2 * operand;
  // Where a row keeps its k-th eight of k (16 bytes): turned so that the same
  // eight of eight rows in a row, which eight lanes read at once, lie in
  // different banks.
  static __host__ __device__ constexpr int at(int row_, int oct) {
    constexpr int octs = stage / 8;
    return row_ * row + 16 * (oct ^ (row_ / (8 / octs) % octs));
  }
};

enum Kind { kForward = 0, kData = 1, kWeights = 2 };

struct SplitArgs {
  const float* x;      // [M, W] (kForward, kWeights)
  const float* dy[2];  // [M, W] per gate (kData, kWeights)
  const float* w[2];   // [H, 256, 256] per gate (kForward, kData)
  float* out[2];       // kForward: [M, W] per gate; kData: [M, W];
                       // kWeights: [H, 256, 256] per gate (one row range)
  const float* bias[2];  // kForward: [W] per gate, or null
  float* part;         // kWeights, several ranges: [splits][2 H][256][256]
  int64_t M;
  int W, H;
  int tiles;           // kForward, kData: of rows
  int splits, rows_per_split;  // kWeights: row ranges
};

// One operand: element (r, k) of its rows (of the result's rows or columns) lies at byte r * row + k * step; elements outside the descriptor are zeros.
struct Source {
  __amdgpu_buffer_rsrc_t base;
  uint32_t row, step;
};

struct Pieces {
  u32x4 hi, mid, lo;  // eight k
};
constexpr float kScale = 0x1p24f;

__device__ __forceinline__ void cut(const float (&v)[8], Pieces& p) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t piece[3];
    cut_bf16x2(v[2 * i], v[2 * i + 1], piece);
    p.hi[i] = piece[0];
    p.mid[i] = piece[1];
    p.lo[i] = piece[2];
  }
}

// A thread's share of one operand's stage: eight k of a row.
template <class S, bool ALONG_K, bool SCALED>
struct Share {
  float v[8];

  static __device__ __forceinline__ int row(int tid) {
    return ALONG_K ? tid / (S::stage / 8) : tid % S::tile;
  }
  static __device__ __forceinline__ int oct(int tid) {
    return ALONG_K ? tid % (S::stage / 8) : tid / S::tile;
  }
  // CHECKED: k may lie outside the operand (the descriptor checks the vector
  // part of an offset, not the scalar one)
  template <bool CHECKED>
  __device__ __forceinline__ void request(const Source& s, uint32_t k0,
                                          int tid) {
    const uint32_t lane_at =
        (uint32_t)row(tid) * s.row + 8u * (uint32_t)oct(tid) * s.step;
    auto word = [&](uint32_t k) {
      return __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(
                     s.base, lane_at + (CHECKED ? k * s.step : 0u),
                     CHECKED ? 0u : k * s.step, 0));
    };
    if constexpr (ALONG_K) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f32x4 t = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(s.base, lane_at + 16u * q,
                                                         k0 * s.step, 0));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[4 * q + i] = t[i];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = word(k0 + (uint32_t)k);
    }
  }
  __device__ __forceinline__ void store(unsigned char* lds, int tid) {
    unsigned char* const at = lds + S::at(row(tid), oct(tid));
    if (SCALED) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] *= kScale;
    }
    Pieces p;
    cut(v, p);
    *reinterpret_cast<u32x4*>(at) = p.hi;
    *reinterpret_cast<u32x4*>(at + S::piece) = p.mid;
    *reinterpret_cast<u32x4*>(at + 2 * S::piece) = p.lo;
  }
};

union Frag {
  u32x4 u;
  bf16x8 v;
};

template <int KIND, int BLOCKS>
__global__ void __launch_bounds__(kThreads, BLOCKS == 1 ? 3 : 2)
gates_split_f32_kernel(SplitArgs p) {
  using S = Size<BLOCKS>;
  constexpr int kTile = S::tile, kStage = S::stage;
  // operand A gives the results' rows, B their columns
  constexpr bool kAlongKA = KIND != kWeights, kAlongKB = KIND == kData;
  // operands cut kScale times as large
  constexpr bool kScaledA = KIND != kForward, kScaledB = KIND == kWeights;
  constexpr float kBack = (kScaledA ? 1.0f / kScale : 1.0f) *
                          (kScaledB ? 1.0f / kScale : 1.0f);
  __shared__ __align__(16) unsigned char lds[2 * S::buffer];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Workgroups go to the eight XCDs in turn: those that share rows of x or dy,
  // or a head's weights, are dealt to one XCD.
  int id = blockIdx.x;
  {
    const int per_xcd = (int)gridDim.x / 8;
    if (id < 8 * per_xcd) id = (id & 7) * per_xcd + (id >> 3);
  }
  const uint32_t row_bytes = (uint32_t)p.W * 4u;
  const uint32_t head_row = kBW * 4u;  // of a head's weights
  constexpr uint32_t head_bytes = kBW * kBW * 4u;
  Source a, b;
  __amdgpu_buffer_rsrc_t a2, b2;  // kData: the recurrence gate's
  int64_t m0 = 0;
  int head, gate = 0, i0 = 0, j0 = 0, split = 0;
  uint32_t rows = 0;    // of this workgroup's range (kWeights: along k)
  uint32_t k_total;
  if constexpr (KIND == kWeights) {
    constexpr int kSide = kBW / kTile, kParts = 2 * kSide * kSide;
    const int which = id % kParts;
    gate = which / (kSide * kSide);
    i0 = which % kSide * kTile;
    j0 = which / kSide % kSide * kTile;
    head = id / kParts % p.H;
    split = id / kParts / p.H;
    m0 = (int64_t)split * p.rows_per_split;
    int64_t left = p.M - m0;
    if (left > p.rows_per_split) left = p.rows_per_split;
    rows = left > 0 ? (uint32_t)left : 0u;
    a = {make_rsrc(p.x + m0 * p.W + head * kBW + i0,
                   rows ? (rows - 1) * row_bytes + kTile * 4u : 0),
         4u, row_bytes};
    b = {make_rsrc((gate ? p.dy[1] : p.dy[0]) + m0 * p.W + head * kBW + j0,
                   rows ? (rows - 1) * row_bytes + kTile * 4u : 0),
         4u, row_bytes};
    k_total = rows;
  } else {
    constexpr int kSide = kBW / kTile;  // parts of a gate's results
    constexpr int kParts = KIND == kForward ? 2 * kSide : kSide;
    const int part = id % kParts;
    const int tile = id / kParts % p.tiles;
    head = id / kParts / p.tiles;
    gate = part / kSide;
    j0 = part % kSide * kTile;
    m0 = (int64_t)tile * kTile;
    const int64_t left = p.M - m0;
    rows = (uint32_t)(left < kTile ? left : kTile);
    // (a descriptor ends with the last row's part of this head)
    const uint32_t bytes = (rows - 1) * row_bytes + kBW * 4u;
    if constexpr (KIND == kForward) {
      a = {make_rsrc(p.x + m0 * p.W + head * kBW, bytes), row_bytes, 4u};
      b = {make_rsrc((gate ? p.w[1] : p.w[0]) + (int64_t)head * kBW * kBW + j0,
                     head_bytes - 4u * (uint32_t)j0),
           4u, head_row};
      k_total = kBW;
    } else {
      a = {make_rsrc(p.dy[0] + m0 * p.W + head * kBW, bytes), row_bytes, 4u};
      a2 = make_rsrc(p.dy[1] + m0 * p.W + head * kBW, bytes);
      const int64_t at = ((int64_t)head * kBW + j0) * kBW;
      b = {make_rsrc(p.w[0] + at, kTile * head_row), head_row, 4u};
      b2 = make_rsrc(p.w[1] + at, kTile * head_row);
      k_total = 2 * kBW;
    }
  }

  // Two stages of both operands in flight: a stage's floats are requested two
  // stages ahead and cut during the one before it, between its matrix
  // instructions.
  Share<S, kAlongKA, kScaledA> sa[2];
  Share<S, kAlongKB, kScaledB> sb[2];
  auto request = [&](uint32_t k, auto SLOT) {
    constexpr int slot = decltype(SLOT)::value;
    constexpr bool checked = KIND == kWeights;
    // (past the last stage: the first again, or zeros)
    if (!checked) k &= k_total - 1;
    const bool second = KIND == kData && k >= kBW;
    if (second) k -= kBW;
    const Source qa = {second ? a2 : a.base, a.row, a.step};
    const Source qb = {second ? b2 : b.base, b.row, b.step};
    sa[slot].template request<checked>(qa, k, tid);
    sb[slot].template request<checked>(qb, k, tid);
  };
  // this wave's results
  const int wr = kTile / 2 * (wave >> 1), wc = kTile / 2 * (wave & 1);
  f32x16 big[BLOCKS][BLOCKS], small[BLOCKS][BLOCKS];
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) big[i][j][r] = small[i][j][r] = 0.0f;
  // this lane's eight k of its row in the first block, per 16 k of a stage
  const unsigned char* la[kStage / 16];
  const unsigned char* lb[kStage / 16];
#pragma unroll
  for (int ks = 0; ks < kStage / 16; ++ks) {
    la[ks] = lds + S::at(wr + (lane & 31), 2 * ks + (lane >> 5));
    lb[ks] = lds + S::operand + S::at(wc + (lane & 31), 2 * ks + (lane >> 5));
  }
  // Stage k from buffer SLOT; the next one's floats are cut into the other
  // buffer, and their registers take what is asked for of the stage after the
  // one after it.
  auto stage = [&](uint32_t k, auto SLOT) {
    constexpr int slot = decltype(SLOT)::value;
    unsigned char* const other = lds + (slot ^ 1) * S::buffer;
#pragma unroll
    for (int ks = 0; ks < kStage / 16; ++ks) {
      const bool first = ks == 0, last = ks == kStage / 16 - 1;
      Frag fa[BLOCKS][3], fb[BLOCKS][3];
      auto pieces = [&](int q) {
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) {
          const int at = slot * S::buffer + q * S::piece + 32 * i * S::row;
          fa[i][q].u = *reinterpret_cast<const u32x4*>(la[ks] + at);
          fb[i][q].u = *reinterpret_cast<const u32x4*>(lb[ks] + at);
        }
      };
      auto multiply = [&](f32x16 (&sum)[BLOCKS][BLOCKS], int qa, int qb) {
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
          for (int j = 0; j < BLOCKS; ++j)
            sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                fa[i][qa].v, fb[j][qb].v, sum[i][j], 0, 0, 0);
      };
      pieces(0);
      pieces(1);
      multiply(big, 0, 0);
      if (first) sa[slot ^ 1].store(other, tid);
      multiply(small, 0, 1);
      __builtin_amdgcn_sched_barrier(0);
      pieces(2);
      multiply(small, 1, 0);
      if (last) sb[slot ^ 1].store(other + S::operand, tid);
      multiply(small, 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      if (last)
        request(k + 3 * kStage, std::integral_constant<int, slot ^ 1>{});
      multiply(small, 0, 2);
      multiply(small, 2, 0);
    }
    lds_barrier();
  };
  request(0, std::integral_constant<int, 0>{});
  request(kStage, std::integral_constant<int, 1>{});
  sa[0].store(lds, tid);
  sb[0].store(lds + S::operand, tid);
  request(2 * kStage, std::integral_constant<int, 0>{});
  lds_barrier();
  for (uint32_t k = 0; k < k_total; k += 2 * kStage) {
    stage(k, std::integral_constant<int, 0>{});
    // (an odd number of stages ends with one of zeros)
    stage(k + kStage, std::integral_constant<int, 1>{});
  }

  float odd = 0.0f;  // NaN as soon as one result is not finite
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float sum = big[i][j][r] + small[i][j][r];
        odd = __builtin_fmaf(sum, 0.0f, odd);
        big[i][j][r] = sum * kBack;
      }
  if (__builtin_expect(__any(odd != 0.0f), 0)) {
    // infinities, NaN or an overflow: the float32 instruction instead
    auto element = [&](__amdgpu_buffer_rsrc_t base, const Source& s, uint32_t r,
                       uint32_t k) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           base, r * s.row + k * s.step, 0, 0));
    };
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int j = 0; j < BLOCKS; ++j) {
        f32x16 again;
#pragma unroll
        for (int r = 0; r < 16; ++r) again[r] = 0.0f;
        const uint32_t ra = (uint32_t)(wr + 32 * i + (lane & 31));
        const uint32_t rb = (uint32_t)(wc + 32 * j + (lane & 31));
        for (uint32_t k = 0; k < k_total; k += 2) {
          const bool second = KIND == kData && k >= kBW;
          const uint32_t kk = (second ? k - kBW : k) + (uint32_t)(lane >> 5);
          const float va = element(second ? a2 : a.base, a, ra, kk);
          const float vb = element(second ? b2 : b.base, b, rb, kk);
          again = __builtin_amdgcn_mfma_f32_32x32x2f32(va, vb, again, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (big[i][j][r] * 0.0f != 0.0f) big[i][j][r] = again[r];
      }
  }

  // block (i, j), result r of a lane: row 8 (r / 4) + 4 (lane / 32) + r % 4,
  // column lane % 32
  if constexpr (KIND == kWeights) {
    float* const dst =
        (p.splits == 1
             ? (gate ? p.out[1] : p.out[0]) + (int64_t)head * kBW * kBW
             : p.part + ((int64_t)split * 2 * p.H + gate * p.H + head) * kBW *
                            kBW) +
        (i0 + wr) * kBW + j0 + wc + (lane & 31);
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
#pragma unroll
        for (int j = 0; j < BLOCKS; ++j) dst[row * kBW + 32 * j] = big[i][j][r];
      }
  } else {
    // (rows past the end fall outside the descriptor)
    const __amdgpu_buffer_rsrc_t ro =
        make_rsrc((gate ? p.out[1] : p.out[0]) + m0 * p.W, rows * row_bytes);
    const uint32_t at = (uint32_t)(wr + 4 * (lane >> 5)) * row_bytes +
                        4u * (uint32_t)(head * kBW + j0 + wc + (lane & 31));
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int j = 0; j < BLOCKS; ++j) {
        float bias = 0.0f;
        if (KIND == kForward && p.bias[0])
          bias = (gate ? p.bias[1] : p.bias[0])[head * kBW + j0 + wc + 32 * j +
                                                (lane & 31)];
        float before[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t off =
              at + (uint32_t)(32 * i + 8 * (r >> 2) + (r & 3)) * row_bytes +
              128u * j;
          before[r] = 0.0f;
          if (KIND == kData)
            before[r] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(ro, off, 0, 0));
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t off =
              at + (uint32_t)(32 * i + 8 * (r >> 2) + (r & 3)) * row_bytes +
              128u * j;
          const float v =
              KIND == kData ? before[r] + big[i][j][r] : big[i][j][r] + bias;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ro, off, 0, 0);
        }
      }
  }
}

// Adds the row ranges' sums in their order.
__global__ void __launch_bounds__(256)
gates_wgrad_finish_kernel(const f32x4* __restrict__ part, int splits,
                          int64_t items, f32x4* __restrict__ dwx,
                          f32x4* __restrict__ dwa) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= 2 * items) return;
  f32x4 v = part[e];
  for (int s = 1; s < splits; ++s) {
    const f32x4 w = part[(int64_t)s * 2 * items + e];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] += w[k];
  }
  if (e < items) dwx[e] = v;
  else dwa[e - items] = v;
}

int splits_for(int64_t M, int H) {
  // as many row ranges as keep every workgroup resident, two to a CU; at least
  // 128 rows each
  int64_t want = 512 / ((int64_t)8 * H);
  const int64_t most = (M + 127) / 128;
  if (want > most) want = most;
  return want < 1 ? 1 : (int)want;
}

int64_t rows_for(int64_t M, int splits) {
  const int64_t rows = (M + splits - 1) / splits;
  return (rows + 31) / 32 * 32;  // (two stages)
}

template <int KIND, int BLOCKS>
hipError_t launch(SplitArgs& a, hipStream_t s) {
  using S = Size<BLOCKS>;
  const int64_t side = kBW / S::tile;
  int64_t blocks;
  if (KIND == kWeights) {
    blocks = a.H * a.splits * 2 * side * side;
  } else {
    a.tiles = (int)((a.M + S::tile - 1) / S::tile);
    blocks = (int64_t)a.tiles * a.H * side * (KIND == kForward ? 2 : 1);
  }
  if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
  gates_split_f32_kernel<KIND, BLOCKS>
      <<<dim3((unsigned)blocks), kThreads, 0, s>>>(a);
  return hipGetLastError();
}

// Tiles of 64 x 64 while their workgroups, four for one of 128 x 128, are all
// resident (three to a CU): us, 64 / 128, forward 10 heads 64 rows 8 / 15, 333 rows
// (480 workgroups) 12 / 17, 512 (640) 14.9 / 17.1, 768 (960) 19.6 / 18.7; 16 heads
// 333 rows (768) 15 / 17, 1001 (2048) 35 / 28; data 10 heads 768 rows (480) 18 / 26,
// 1500 (960) 34 / 29.  Same products in the same order: the same bits.
template <int KIND>
hipError_t launch_rows(SplitArgs& a, hipStream_t s) {
  const int64_t small =
      (a.M + 63) / 64 * a.H * (KIND == kForward ? 8 : 4);
  if (small <= 768) return launch<KIND, 1>(a, s);
  return launch<KIND, 2>(a, s);
}

}  // namespace

bool gates_f32_serves(int64_t M, int W, int H) {
  // (128 rows of an operand are 32-bit offsets)
  return M > 0 && H > 0 && H <= 4096 && W == H * kBW &&
         (M + 63) / 64 * H * 8 <= 0x7fffffff;
}

hipError_t launch_gates_f32(const void* x, const void* w_x, const void* w_a,
                            const void* b_x, const void* b_a, void* gx, void* ga,
                            int64_t M, int W, int H, hipStream_t s) {
  if (!gates_f32_serves(M, W, H)) return hipErrorInvalidValue;
  SplitArgs a{};
  a.bias[0] = (const float*)b_x;
  a.bias[1] = (const float*)b_a;
  a.x = (const float*)x;
  a.w[0] = (const float*)w_x;
  a.w[1] = (const float*)w_a;
  a.out[0] = (float*)gx;
  a.out[1] = (float*)ga;
  a.M = M;
  a.W = W;
  a.H = H;
  return launch_rows<kForward>(a, s);
}

hipError_t launch_gates_dgrad_f32(const void* dgx, const void* dga,
                                  const void* w_x, const void* w_a, void* dx,
                                  int64_t M, int W, int H, hipStream_t s) {
  if (!gates_f32_serves(M, W, H)) return hipErrorInvalidValue;
  SplitArgs a{};
  a.dy[0] = (const float*)dgx;
  a.dy[1] = (const float*)dga;
  a.w[0] = (const float*)w_x;
  a.w[1] = (const float*)w_a;
  a.out[0] = (float*)dx;
  a.M = M;
  a.W = W;
  a.H = H;
  return launch_rows<kData>(a, s);
}

bool gates_wgrad_f32_serves(int64_t M, int W, int H) {
  if (M <= 0 || H <= 0 || W != H * kBW || H > 4096) return false;
  // offsets within a row range, a stage past its end, are 32 bits
  return (uint64_t)(rows_for(M, splits_for(M, H)) + 64) * (uint64_t)W *
             4u < 0xffffffffull;
}

size_t gates_wgrad_f32_workspace_bytes(int64_t M, int W, int H) {
  const int splits = splits_for(M, H);
  return splits == 1 ? 0 : (size_t)splits * 2 * H * kBW * kBW * sizeof(float);
}

hipError_t launch_gates_wgrad_f32(const void* x, const void* dgx,
                                  const void* dga, void* dwx, void* dwa,
                                  void* workspace, int64_t M, int W, int H,
                                  hipStream_t s) {
  if (!gates_wgrad_f32_serves(M, W, H)) return hipErrorInvalidValue;
  SplitArgs a{};
  a.x = (const float*)x;
  a.dy[0] = (const float*)dgx;
  a.dy[1] = (const float*)dga;
  a.out[0] = (float*)dwx;
  a.out[1] = (float*)dwa;
  a.part = (float*)workspace;
  a.M = M;
  a.W = W;
  a.H = H;
  a.splits = splits_for(M, H);
  a.rows_per_split = (int)rows_for(M, a.splits);
  hipError_t e = launch<kWeights, 2>(a, s);
  if (e != hipSuccess || a.splits == 1) return e;
  const int64_t items = (int64_t)H * kBW * kBW / 4;
  gates_wgrad_finish_kernel<<<dim3((unsigned)((2 * items + 255) / 256)), 256, 0,
                              s>>>((const f32x4*)workspace, a.splits, items,
                                   (f32x4*)dwx, (f32x4*)dwa);
  return hipGetLastError();
}

}  // namespace rg
