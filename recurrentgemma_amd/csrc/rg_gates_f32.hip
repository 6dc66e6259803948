// The two gate projections of RGLRU.forward in float32 (256-wide heads) for
// the differentiable path, without their biases
// (recurrentgemma/torch/layers.py:127-137, called twice on the same x at
// :338-339):  y_g[m, h, j] = sum_i x[m, h, i] w_g[h, i, j].
//
// Bound by the matrix pipe (v_mfma_f32_32x32x2_f32, 64 cycles each): the
// operands go from memory to registers without LDS.  A lane of the instruction
// holds one value, row (or column) lane % 32 of k lane / 32; which two k an
// instruction takes is free, so lane l loads four consecutive k,
// 8 s + 4 (l / 32) .. + 3, of its row of x with 16 bytes and has the operand of
// four instructions, and four consecutive columns 4 (l % 32) .. + 3 of one k of
// the weights: the operands of four column blocks, and four consecutive
// columns of a result row, stored as 16 bytes.  Per eight k a wave issues five
// loads for 16 matrix instructions, two such steps ahead.
//
// A wave has 32 rows by 128 columns, a workgroup's four waves are the column
// halves of both gates on the same rows.  Consecutive workgroups of an XCD
// share a head, whose weights (512 KB) stay in its L2.  The two halves of the
// 256 k are summed apart: half as long a chain of roundings.
//
// Measured against the library's two batched products on strided views (its
// tiles of 256 rows leave the chip idle or with a short last round), us, and
// the error against 64 bits, 2.0e-7 here and 2.9e-7 there:
//   rows                  64    200    512   1001   2048   3003   5000   8192
//   width 2560, here      18     19     21     37     54     72    122    182
//               library   37    129     33     50     82     79    143    188
//   width 4096, here      18     20     24     42     74    102    172    291
//               library   37    130     27     47     82    145    184    292
// 64 rows a wave (half the loads of weights per product) is 8 % ahead from 1024
// workgroups on (255 us at 8192 x 4096) and behind below, but leaves no
// registers for the second half's sums.  The backward of x in the same form
// (weights read down their rows) was behind the library's and is not here.
#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kBW = 256;
constexpr int kSteps = kBW / 8;  // of eight k
constexpr int kRows = 32;

struct GatesF32Args {
  const float* x;     // [M, W]
  const float* w[2];  // [H, 256, 256]
  float* y[2];        // [M, W]
  int64_t M;
  int W, H;
  int tiles;          // of kRows rows
};

struct Operands {
  f32x4 a;
  f32x4 b[4];
};

__global__ void __launch_bounds__(256, 2) gates_f32_kernel(GatesF32Args p) {
  const int lane = threadIdx.x & 63, half = lane >> 5, n = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int id = blockIdx.x;
  {
    const int per_xcd = (int)gridDim.x / 8;
    if (id < 8 * per_xcd) id = (id & 7) * per_xcd + (id >> 3);
  }
  const int head = id / p.tiles;
  const int gate = wave >> 1, c0 = (wave & 1) * 128;
  const int64_t m0 = (int64_t)(id % p.tiles) * kRows;
  const int64_t left = p.M - m0;

  // descriptors over this tile's rows: the others read as zeros, their stores
  // are dropped
  const uint32_t row_bytes = (uint32_t)p.W * 4u;
  const uint32_t span = (uint32_t)(left < kRows ? left : kRows) * row_bytes;
  const uint32_t head_at = (uint32_t)head * (kBW * 4u);
  const uint32_t at_x = (uint32_t)n * row_bytes + head_at + 16u * half;
  const uint32_t at_w = (uint32_t)(4 * half) * (kBW * 4u) + 4u * (c0 + 4 * n);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x + m0 * p.W, span);
  const __amdgpu_buffer_rsrc_t rw =
      make_rsrc((gate ? p.w[1] : p.w[0]) + (int64_t)head * kBW * kBW,
                kBW * kBW * 4u);
  auto request = [&](int step, Operands& t) {
    const uint32_t s = (uint32_t)step & (kSteps - 1);  // (past the end: again)
    t.a = __builtin_bit_cast(
        f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, at_x + 32u * s, 0, 0));
#pragma unroll
    for (int q = 0; q < 4; ++q)
      t.b[q] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     rw, at_w + (8u * s + (uint32_t)q) * (kBW * 4u), 0, 0));
  };
  f32x16 acc[2][4];  // per half of k and column block
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[k][d][r] = 0.0f;
  auto multiply = [&](const Operands& t, f32x16 (&sum)[4]) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int d = 0; d < 4; ++d)
        sum[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(t.a[c], t.b[c][d], sum[d],
                                                      0, 0, 0);
  };
  Operands even, odd;
  request(0, even);
  request(1, odd);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    for (int s = k * (kSteps / 2); s < (k + 1) * (kSteps / 2); s += 2) {
      multiply(even, acc[k]);
      request(s + 2, even);
      __builtin_amdgcn_sched_barrier(0);
      multiply(odd, acc[k]);
      request(s + 3, odd);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  const __amdgpu_buffer_rsrc_t ry =
      make_rsrc((gate ? p.y[1] : p.y[0]) + m0 * p.W, span);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t row = 8 * (r >> 2) + 4 * half + (r & 3);
    f32x4 v;
#pragma unroll
    for (int d = 0; d < 4; ++d) v[d] = acc[0][d][r] + acc[1][d][r];
    __builtin_amdgcn_raw_buffer_store_b128(
        __builtin_bit_cast(u32x4, v), ry,
        row * row_bytes + head_at + 4u * (c0 + 4 * n), 0, 0);
  }
}

}  // namespace

bool gates_f32_serves(int64_t M, int W, int H) {
  return M > 0 && H > 0 && H <= 32768 && W == H * kBW &&
         (M + kRows - 1) / kRows * H <= 0x7fffffff;
}

hipError_t launch_gates_f32(const void* x, const void* w_x, const void* w_a,
                            void* gx, void* ga, int64_t M, int W, int H,
                            hipStream_t s) {
  if (!gates_f32_serves(M, W, H)) return hipErrorInvalidValue;
  const int64_t tiles = (M + kRows - 1) / kRows;
  const GatesF32Args a{(const float*)x,
                       {(const float*)w_x, (const float*)w_a},
                       {(float*)gx, (float*)ga},
                       M, W, H, (int)tiles};
  gates_f32_kernel<<<dim3((unsigned)(tiles * H)), 256, 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace rg
