// Weight gradients of both gate projections of RGLRU.forward in float32
// (256-wide heads): what autograd forms for
//   y[m, h, j] = sum_i x[m, h, i] w[h, i, j]
// (recurrentgemma/torch/layers.py:127-137, called twice on the same x at
// :338-339) from the gradients dy of the two outputs:
//   dw[h, i, j] = sum_m x[m, h, i] dy[m, h, j].
//
// Bound by the matrix pipe: v_mfma_f32_32x32x2_f32 takes 64 cycles, so
// everything else is there to keep one issued after the other.  Its operands
// are one value per lane (32 channels x 2 m), which a row of x or dy gives
// without any transposition, and which channel sits in which lane is free:
// lane l takes channels 4 l .. 4 l + 3 of 128 (one 16-byte load, the four
// values are the A operands of four blocks) and 2 l, 2 l + 1 of 64 (one 8-byte
// load, two B operands).  Two loads feed eight matrix instructions, straight
// from memory to registers: no LDS in the loop.
//
// A workgroup owns a 128 x 64 tile of one head's dw for one gate and a range
// of rows m; its four waves take batches of eight rows in turn, two batches
// (48 registers) requested ahead, and are added through LDS at the end.  Row
// ranges as long as two workgroups a CU (the accumulators take half of the
// registers) are all resident; their sums are added in a fixed order by a
// second kernel, so results do not vary from run to run.
//
// Measured against the library's two batched products on strided views, us, and
// the error of dw against 64 bits (a wave's chain of sums is a quarter of a row
// range; the second kernel, 5 us of these, included):
//   rows                  512    1001    2048    3003    4096    8192   16384
//   10 heads, here         26      38      59      73      96     180     356
//             library     239     456     106     133     143     313     741
//             error    1.3e-7  1.7e-7  2.4e-7  2.9e-7  3.4e-7  4.7e-7  6.6e-7
//             library  4.1e-7  5.7e-7  8.1e-7  9.2e-7  1.1e-6  1.6e-6  2.2e-6
//   16 heads, here         32      47      81     104     135     270     529
//             library     238     456      74      98     126     246     506
//             error    1.5e-7  2.1e-7  2.9e-7  3.5e-7  4.1e-7  5.7e-7  8.1e-7
//             library  4.1e-7  5.7e-7  8.1e-7  9.8e-7  1.2e-6  1.6e-6  2.3e-6
// 1 to 4 heads 1.5 to 30 times as fast; 32 heads within 10 % from 2048 rows on.
// 3003 rows of 10 heads are 108 TFLOP/s of the fp32 matrix peak's 157.
#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kBW = 256;            // head width
constexpr int kTileI = 128, kTileJ = 64;
constexpr int kTiles = (kBW / kTileI) * (kBW / kTileJ);  // of a head and gate
constexpr int kWaves = 4;
constexpr int kBatch = 8;           // rows a wave takes at a time
constexpr int kStep = kWaves * kBatch;

struct WgradF32Args {
  const float* x;       // [M, W]
  const float* dy[2];   // [M, W] per gate
  float* dw[2];         // [H, 256, 256] per gate (one row range)
  float* part;          // [splits][2 H][256][256] (several)
  int64_t M;
  int W, H;
  int splits;
  int rows_per_split;   // a multiple of kStep
};

struct Batch {
  f32x4 a[kBatch / 2];
  f32x2 b[kBatch / 2];
};

__global__ void __launch_bounds__(kWaves * 64, 2)
gates_wgrad_f32_kernel(WgradF32Args p) {
  __shared__ float sums[kWaves][32][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The 16 workgroups of a (head, row range) read the same rows: dealt to one
  // XCD (linear id modulo 8), they come from memory once.  The grid is rounded
  // up to whole rounds of eight groups and the surplus exits.
  const int in_xcd = blockIdx.x >> 3;
  const int group = in_xcd / (2 * kTiles) * 8 + (int)(blockIdx.x & 7);
  if (group >= p.H * p.splits) return;
  const int which = in_xcd % (2 * kTiles);
  const int gate = which / kTiles;
  const int i0 = which % 2 * kTileI, j0 = which / 2 % (kBW / kTileJ) * kTileJ;
  const int head = group % p.H, split = group / p.H;
  const int64_t m0 = (int64_t)split * p.rows_per_split;
  int64_t rows = p.M - m0;
  if (rows > p.rows_per_split) rows = p.rows_per_split;
  if (rows < 0) rows = 0;

  // descriptors over the range's rows: those behind it read as zeros
  const uint32_t row_bytes = (uint32_t)p.W * 4u;
  const __amdgpu_buffer_rsrc_t ra =
      make_rsrc(p.x + m0 * p.W, (uint32_t)rows * row_bytes);
  const __amdgpu_buffer_rsrc_t rb =
      make_rsrc(p.dy[gate] + m0 * p.W, (uint32_t)rows * row_bytes);
  const uint32_t first =
      ((uint32_t)(wave * kBatch) + (uint32_t)(lane >> 5)) * row_bytes;
  const uint32_t at_a =
      first + 4u * (uint32_t)(head * kBW + i0 + 4 * (lane & 31));
  const uint32_t at_b =
      first + 4u * (uint32_t)(head * kBW + j0 + 2 * (lane & 31));
  auto request = [&](uint32_t k, Batch& t) {
    const uint32_t base = k * kStep * row_bytes;
#pragma unroll
    for (int s = 0; s < kBatch / 2; ++s) {
      const uint32_t off = base + 2u * s * row_bytes;
      t.a[s] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, at_a + off, 0, 0));
      t.b[s] = __builtin_bit_cast(
          f32x2, __builtin_amdgcn_raw_buffer_load_b64(rb, at_b + off, 0, 0));
    }
  };
  f32x16 acc[4][2];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[c][d][r] = 0.0f;
  auto multiply = [&](const Batch& t) {
#pragma unroll
    for (int s = 0; s < kBatch / 2; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int d = 0; d < 2; ++d)
          acc[c][d] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              t.a[s][c], t.b[s][d], acc[c][d], 0, 0, 0);
  };
  const uint32_t batches = (uint32_t)((rows + kStep - 1) / kStep);
  Batch even, odd;
  request(0, even);
  request(1, odd);
  for (uint32_t k = 0; k < batches; k += 2) {
    multiply(even);
    request(k + 2, even);
    __builtin_amdgcn_sched_barrier(0);
    multiply(odd);  // (behind the last batch: zeros)
    request(k + 3, odd);
    __builtin_amdgcn_sched_barrier(0);
  }

  // Block (c, d), row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32 of a
  // wave's result is channel 4 row + c by channel 2 column + d.
  float* const dst =
      p.splits == 1
          ? p.dw[gate] + (int64_t)head * kBW * kBW
          : p.part + ((int64_t)split * 2 * p.H + gate * p.H + head) * kBW * kBW;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (c) __syncthreads();
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) sums[wave][16 * d + r][lane] = acc[c][d][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = 4 * wave + q;
      f32x2 v;
#pragma unroll
      for (int d = 0; d < 2; ++d)
        v[d] = (sums[0][16 * d + r][lane] + sums[1][16 * d + r][lane]) +
               (sums[2][16 * d + r][lane] + sums[3][16 * d + r][lane]);
      const int i = i0 + 4 * (8 * wave + 4 * (lane >> 5) + q) + c;
      *reinterpret_cast<f32x2*>(dst + i * kBW + j0 + 2 * (lane & 31)) = v;
    }
  }
}

// Adds the row ranges' sums in their order.
__global__ void __launch_bounds__(256)
gates_wgrad_f32_finish_kernel(const f32x4* __restrict__ part, int splits,
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
  // four batches a wave
  int64_t want = 512 / ((int64_t)2 * kTiles * H);
  const int64_t most = (M + 4 * kStep - 1) / (4 * kStep);
  if (want > most) want = most;
  return want < 1 ? 1 : (int)want;
}

int64_t rows_for(int64_t M, int splits) {
  const int64_t rows = (M + splits - 1) / splits;
  return (rows + kStep - 1) / kStep * kStep;
}

}  // namespace

// Every shape it can address: from 16 heads and 2048 rows on the library is ahead
// by up to 10 % (the table above), at three times the error, which is what is
// paid for there.
bool gates_wgrad_f32_serves(int64_t M, int W, int H) {
  if (M <= 0 || H <= 0 || W != H * kBW || H > 4096) return false;
  // offsets within a row range, two batches past its end, are 32 bits
  return (uint64_t)(rows_for(M, splits_for(M, H)) + 4 * kStep) * (uint64_t)W * 4u <
         0xffffffffull;
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
  WgradF32Args a{};
  a.x = (const float*)x;
  a.dy[0] = (const float*)dgx;
  a.dy[1] = (const float*)dga;
  a.dw[0] = (float*)dwx;
  a.dw[1] = (float*)dwa;
  a.part = (float*)workspace;
  a.M = M;
  a.W = W;
  a.H = H;
  a.splits = splits_for(M, H);
  a.rows_per_split = (int)rows_for(M, a.splits);
  const int64_t rounds = ((int64_t)H * a.splits + 7) / 8;
  gates_wgrad_f32_kernel<<<dim3((unsigned)(rounds * 8 * 2 * kTiles)),
                           kWaves * 64, 0, s>>>(a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits == 1) return e;
  const int64_t items = (int64_t)H * kBW * kBW / 4;
  gates_wgrad_f32_finish_kernel<<<dim3((unsigned)((2 * items + 255) / 256)), 256,
                                  0, s>>>((const f32x4*)workspace, a.splits,
                                          items, (f32x4*)dwx, (f32x4*)dwa);
  return hipGetLastError();
}

}  // namespace rg
