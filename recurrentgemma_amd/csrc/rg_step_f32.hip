// Decode step of the recurrent core in one launch, float32 and 256-wide heads: conv step
// from the carried conv state, both gate projections, gate arithmetic, one recurrence
// step, the block's join.  Replaces Conv1D.forward's decode branch
// (recurrentgemma/torch/layers.py:469-474, 491-529) and RGLRU.forward with T == 1
// (layers.py:313-365, 170-177) like rg_fused.hip's bf16 kernel; as a conv step, a gate
// GEMM and a scan step it was three launches and the pre-activations' way through memory.
//
// A workgroup has a tile of rows (different sequences) and 32 channels of a head: all 256
// channels of the head's conv step go into LDS (each of a head's eight workgroups repeats
// it; the conv state is stored by the one whose channels they are), wave (gate, half of K)
// has its 64 weights a lane in registers and its products on v_mfma_f32_32x32x2_f32, the
// halves and the gates meet in LDS, and every thread finishes four outputs.  Arithmetic
// and order of the sums are those of the three kernels (rg_conv.hip, rg_gemm.hip,
// rg_scan.hip): the same bits.
#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kBW = 256;
constexpr int kStride = kBW + 4;  // floats per LDS row (16 rows: 64 banks)
constexpr int kSlices = 8;        // workgroups of a head
constexpr int kThreads = 256;

// ROWS: of a tile, 8, 16 or 32.  (The matrix instructions take 32, those beyond ROWS as
// LDS has them: no other row sees them.)
template <int ROWS, bool JOIN>
__global__ void __launch_bounds__(kThreads, 2) block_step_f32_kernel(StepF32Args p) {
  __shared__ __align__(16) float rows[32 * kStride];
  __shared__ float sums[4][32][33];  // of (gate, half of K): [row][channel]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The workgroups of a (row tile, head) pair, which read the same rows, to one XCD.
  int id = blockIdx.x;
  {
    const int per_xcd = (int)gridDim.x / 8;
    if (id < 8 * per_xcd) id = (id & 7) * per_xcd + (id >> 3);
  }
  const int slice = id % kSlices;
  const int h = id / kSlices % p.H;
  const int b0 = id / kSlices / p.H * ROWS;
  const int64_t W = p.W;
  const uint32_t row_bytes = (uint32_t)W * 4u;
  const uint32_t here = (uint32_t)(p.B - b0 < ROWS ? p.B - b0 : ROWS);
  // (descriptors over the tile's rows: those past the last read as zeros, and their
  // stores are dropped)
  const auto tile_of = [&](const float* base, uint32_t rows_each) {
    return make_rsrc(base + (int64_t)b0 * rows_each * W,
                     base ? here * rows_each * row_bytes : 0u);
  };
  const __amdgpu_buffer_rsrc_t rx = tile_of(p.x, 1), rcin = tile_of(p.cache_in, 3);

  // ---- loads, in the order in which they are used --------------------------------
  // conv: four channels of every fourth row
  constexpr int kPer = ROWS / 4;
  const uint32_t c = (uint32_t)(h * kBW + 4 * lane);
  f32x4 xv[kPer], st[kPer][3];  // state oldest first
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint32_t row = (uint32_t)(wave + 4 * j);
    xv[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                          rx, row * row_bytes + 4u * c, 0, 0));
#pragma unroll
    for (int k = 0; k < 3; ++k)
      st[j][k] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     rcin, (row * 3u + k) * row_bytes + 4u * c, 0, 0));
  }
  f32x4 taps[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    taps[k] = *reinterpret_cast<const f32x4*>(p.conv_w + k * W + c);
  const f32x4 conv_bias = *reinterpret_cast<const f32x4*>(p.conv_b + c);
  // this lane's weights: k = 128 half + 8 j + 4 g + i at 4 j + i
  const int gate = wave & 1, half = wave >> 1;
  const int col = lane & 31, g = lane >> 5;
  float w[64];
  {
    const __amdgpu_buffer_rsrc_t rw =
        make_rsrc(p.w[gate] + (int64_t)h * kBW * kBW, kBW * kBW * 4);
    const uint32_t at = (uint32_t)((128 * half + 4 * g) * kBW + slice * 32 + col) * 4u;
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[4 * j + i] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(
                       rw, at, (uint32_t)((8 * j + i) * kBW * 4), 0));
  }
  // the outputs this thread finishes: one channel of every eighth row
  constexpr int kOut = ROWS / 8;
  const int n = slice * 32 + (tid & 31);
  const uint32_t ch = (uint32_t)(h * kBW + n);
  const float bias_x = p.b[0][ch], bias_a = p.b[1][ch];
  const float a_param = p.a_param[ch];
  float h_in[kOut], branch[JOIN ? kOut : 1];
  uint32_t seg_lo[kOut], seg_hi[kOut];
  {
    const __amdgpu_buffer_rsrc_t rh = tile_of(p.h_in, 1);
    const uint32_t esize = p.seg_kind == kSegI64 ? 8u : 4u;
    const __amdgpu_buffer_rsrc_t rseg =
        make_rsrc((const char*)p.segpos + (int64_t)b0 * esize, here * esize);
#pragma unroll
    for (int k = 0; k < kOut; ++k) {
      const uint32_t row = (uint32_t)((tid >> 5) + 8 * k);
      h_in[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                              rh, row * row_bytes + 4u * ch, 0, 0));
      seg_lo[k] = __builtin_amdgcn_raw_buffer_load_b32(rseg, row * esize, 0, 0);
      seg_hi[k] = __builtin_amdgcn_raw_buffer_load_b32(
          rseg, esize == 8u ? row * esize + 4u : kBufferOutOfRange, 0, 0);
      if (JOIN)
        branch[k] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(
                       tile_of(p.gate_branch, 1), row * row_bytes + 4u * ch, 0, 0));
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- conv step ------------------------------------------------------------------
  {
    const __amdgpu_buffer_rsrc_t rcout = tile_of(p.cache_out, 3);
    const uint32_t c_out = lane / 8 == slice ? 4u * c : kBufferOutOfRange;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t row = (uint32_t)(wave + 4 * j);
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float acc = __builtin_fmaf(xv[j][e], taps[3][e], conv_bias[e]);
#pragma unroll
        for (int k = 2; k >= 0; --k) acc = __builtin_fmaf(st[j][k][e], taps[k][e], acc);
        o[e] = acc;
      }
      *reinterpret_cast<f32x4*>(rows + row * kStride + 4 * lane) = o;
#pragma unroll
      for (int k = 0; k < 3; ++k)
        buffer_store_16(__builtin_bit_cast(u32x4, k < 2 ? st[j][k + 1] : xv[j]), rcout,
                        c_out + (row * 3u + k) * row_bytes, 0);
    }
  }
  lds_barrier();

  // ---- products -------------------------------------------------------------------
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  const float* const a_lane = rows + col * kStride + 128 * half + 4 * g;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(a_lane + 8 * j);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], w[4 * j + i], acc, 0, 0, 0);
  }
  // result register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (8 * (r >> 2) < ROWS) sums[wave][8 * (r >> 2) + 4 * g + (r & 3)][col] = acc[r];
  lds_barrier();

  // ---- gates, recurrence ------------------------------------------------------------
  const __amdgpu_buffer_rsrc_t rhout = tile_of(p.h_out, 1), ry = tile_of(p.y, 1);
  const float decay = softplus_precise(a_param);
#pragma unroll
  for (int k = 0; k < kOut; ++k) {
    const int row = (tid >> 5) + 8 * k;
    const float gx = (sums[0][row][tid & 31] + sums[2][row][tid & 31]) + bias_x;
    const float ga = (sums[1][row][tid & 31] + sums[3][row][tid & 31]) + bias_a;
    const float gate_x = sigmoid_precise(gx);
    const float log_a = (-8.0f * sigmoid_precise(ga)) * decay;
    float a = expf(log_a);
    float mult = sqrtf(1.0f - expf(2.0f * log_a));
    if ((seg_lo[k] | seg_hi[k]) == 0u) {
      a = 0.0f;
      mult = 1.0f;
    }
    const float xn = (rows[row * kStride + n] * gate_x) * mult;
    const float hn = __builtin_fmaf(a, h_in[k], xn);
    const uint32_t at = (uint32_t)row * row_bytes + 4u * ch;
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(hn), rhout, at, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32(
        __float_as_uint(JOIN ? gelu_mul_f32(hn, branch[JOIN ? k : 0]) : hn), ry, at, 0, 0);
  }
}

template <int ROWS>
void step(const StepF32Args& a, hipStream_t s) {
  const int64_t tiles = ((int64_t)a.B + ROWS - 1) / ROWS;
  const dim3 grid((unsigned)(tiles * a.H * kSlices));
  if (a.gate_branch)
    block_step_f32_kernel<ROWS, true><<<grid, kThreads, 0, s>>>(a);
  else
    block_step_f32_kernel<ROWS, false><<<grid, kThreads, 0, s>>>(a);
}

bool apart(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return !a || !b || x + (uintptr_t)a_bytes <= y || y + (uintptr_t)b_bytes <= x;
}

}  // namespace

// A head's workgroups read what all of them need -- x and the conv state -- while others
// store: nothing that is written may be read, but the state where it lies.
bool block_step_f32_serves(const StepF32Args& a) {
  const int64_t one = (int64_t)a.B * a.W * 4;
  if (a.W != a.H * kBW || 3 * one >= (int64_t)0x7fffffff) return false;
  const struct {
    const void* at;
    int64_t bytes;
  } in[] = {{a.x, one}, {a.cache_in, 3 * one}, {a.gate_branch, one}},
    out[] = {{a.y, one}, {a.cache_out, 3 * one}, {a.h_out, one}};
  for (const auto& o : out)
    for (const auto& i : in)
      if (!apart(o.at, o.bytes, i.at, i.bytes)) return false;
  if (a.h_out != a.h_in && !apart(a.h_out, one, a.h_in, one)) return false;
  return apart(a.y, one, a.h_in, one) && apart(a.cache_out, 3 * one, a.h_in, one) &&
         apart(a.y, one, a.h_out, one) && apart(a.y, one, a.cache_out, 3 * one) &&
         apart(a.h_out, one, a.cache_out, 3 * one);
}

// Rows of a tile: the fewest that one workgroup a CU holds, 8 only for up to 8 rows (9 to
// 16: 6.5 with tiles of 16, 7.1 with two of 8).  What bounds it: launch, loads, 64 matrix
// instructions and the exchange one behind the other for few rows; from two workgroups a
// CU on the matrix pipe (4.2 GFLOP at 512 rows of 4096: 30 us at 142 TFLOP/s) and the
// head's rows, which each of its eight workgroups reads.  us a step, replayed from a graph
// over 4 states, three launches / this:
//   rows              1            8           16           64          173          512
//   width 2560  13.8 /  5.7  15.5 /  5.7  17.7 /  6.6  26.9 /  9.7  37.3 / 16.6  67.5 / 34.6
//   width 4096  15.5 /  6.2  17.5 /  6.4  20.3 /  7.4  29.7 / 10.9  47.8 / 23.7 104.5 / 49.5
// (two workgroups a CU asked for: the compiler keeps tiles of 32 rows within 256 registers,
// else 264; 512 rows of 4096 67 -> 50.)
hipError_t launch_block_step_f32(const StepF32Args& a, hipStream_t s) {
  const int64_t tiles8 = ((int64_t)a.B + 7) / 8;
  if (tiles8 <= 0 || tiles8 * a.H * kSlices > 0x7fffffff) return hipErrorInvalidValue;
  if (a.B <= 8) step<8>(a, s);
  else if ((tiles8 + 1) / 2 * a.H * kSlices <= 256) step<16>(a, s);
  else step<32>(a, s);
  return hipGetLastError();
}

}  // namespace rg
