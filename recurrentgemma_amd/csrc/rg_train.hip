// The parts of a training step's backward pass that are neither the recurrence
// (rg_scan_tiles.hip), the conv (rg_conv.hip), the gates' weight gradients
// (rg_gates_wgrad.hip) nor a library matrix product:
//  * gates_dgrad_kernel: the input gradient of both gate projections added to
//    the one that comes from the recurrence, one pass instead of two
//    block-diagonal products, two sums and two transposed weight copies;
//  * column sums (bias gradients), alone and inside the join's backward pass,
//    as partial sums of 64 rows, and one kernel that finishes several of them.
#include "rg_common.h"
#include "rg_internal.h"
#include "rg_weight_frags.h"

namespace rg {
namespace {

typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) float lds_f32;

// ---- dx += dgx W_x^T + dga W_a^T (autograd of layers.py:127-137) ------------
// A workgroup of eight waves belongs to one head and walks tiles of 64 rows;
// wave w keeps the 512 (both gates' outputs) x 32 (inputs 32 w ..) weights as
// 32 B fragments in accumulation registers: lane (n, k half) needs
// W[n, 8 consecutive k], which is how the reference stores them.  Rows of dgx
// and dga come through the memory pipe into LDS (two tiles, the next one in
// flight), their 16-byte chunks permuted by the row's number so that the
// operand reads of 32 rows meet every bank equally; the results leave through
// an fp32 patch per wave as 16-byte row chunks, added to dx there.
// HBM-bound: 4 tensors, 8 bytes per element (168 MB at M 8192, W 2560).
constexpr int kBW = 256;
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kRows = 64;                   // rows per tile
constexpr int kRowBytes = 2 * kBW * 2;      // dgx and dga of a row
constexpr int kTileBytes = kRows * kRowBytes;
constexpr int kPatchFloats = 36;            // 32 channels + padding
constexpr int kPatchOff = 2 * kTileBytes;
constexpr int kDgradLds = kPatchOff + kWaves * 16 * kPatchFloats * 4;
static_assert(kDgradLds <= 160 * 1024, "LDS of one CU");

__global__ void __launch_bounds__(kThreads)
gates_dgrad_kernel(const uint16_t* __restrict__ dgx,
                   const uint16_t* __restrict__ dga,
                   const uint16_t* __restrict__ w_x,
                   const uint16_t* __restrict__ w_a, uint16_t* dx, int64_t M,
                   int W, int H, int ranges) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  lds_byte* const lds3 = (lds_byte*)lds_raw;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.x % H;
  const int range = blockIdx.x / H;
  const int64_t tiles = (M + kRows - 1) / kRows;

  const uint32_t row_bytes = 2u * (uint32_t)W;
  // rows of one tile -> LDS: a wave-wide load covers one row's 512 bytes of
  // either gate in one half of the lanes each; chunk p of row r holds the
  // row's chunk p ^ (r % 32).  Rows past the end read as zeros.
  auto request = [&](int64_t tile, int buf) {
    const int64_t m0 = tile * kRows;
    const int64_t left = M - m0;
    const uint32_t bytes =
        left <= 0 ? 0u
                  : (uint32_t)(left < kRows ? left : kRows) * row_bytes;
    const int64_t at = left <= 0 ? 0 : m0 * W;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(dgx + at, bytes);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(dga + at, bytes);
#pragma unroll
    for (int j = 0; j < kRows / kWaves / 2; ++j) {
      // two rows of one gate per load: lanes 0-31 row r, lanes 32-63 row r + 1
      const int r = 2 * (wave + kWaves * j);
      const int row = r + (lane >> 5);
      const uint32_t chunk = (uint32_t)((lane & 31) ^ (row & 31));
      const uint32_t off =
          (uint32_t)row * row_bytes + 2u * (uint32_t)(h * kBW) + 16u * chunk;
      lds_byte* const dst = lds3 + buf * kTileBytes + r * (kBW * 2);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, dst, 16, off, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ra, dst + kRows * kBW * 2, 16, off, 0, 0, 0);
    }
  };
  int64_t tile = range;
  int buf = 0;
  request(tile, 0);
  // weights: fragment f = 16 gate + k-step
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const uint16_t* src = (half ? w_a : w_x) +
                          ((int64_t)h * kBW + 32 * wave + (lane & 31)) * kBW +
                          8 * (lane >> 5);
    f32x4 w[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
      w[k] = *reinterpret_cast<const f32x4*>(src + 16 * k);
    asm volatile("" ::"v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]),
                 "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]),
                 "v"(w[10]), "v"(w[11]), "v"(w[12]), "v"(w[13]), "v"(w[14]),
                 "v"(w[15]));
#pragma unroll
    for (int k = 0; k < 16; ++k) set_weight_frag(16 * half + k, w[k]);
  }
  const uint32_t patch = kPatchOff + wave * 16 * kPatchFloats * 4;
  for (; tile < tiles; tile += ranges, buf ^= 1) {
    // this tile's rows are in LDS (every wave waits for its own loads), and
    // nobody reads the other buffer any more
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (tile + ranges < tiles) request(tile + ranges, buf ^ 1);
    const int64_t m0 = tile * kRows;
    const int64_t left = M - m0;
    const __amdgpu_buffer_rsrc_t rdx = make_rsrc(
        dx + m0 * W, (uint32_t)(left < kRows ? left : kRows) * row_bytes);
#pragma unroll
    for (int rh = 0; rh < 2; ++rh) {  // rows 32 rh .. 32 rh + 31
      const uint32_t off = (uint32_t)(32 * rh + (lane >> 2)) * row_bytes +
                           2u * (uint32_t)(h * kBW + 32 * wave) + 16u * (lane & 3);
      // what is there already, 16 rows at a time
      u32x4 old[2];
#pragma unroll
      for (int g = 0; g < 2; ++g)
        old[g] = __builtin_amdgcn_raw_buffer_load_b128(
            rdx, off + 16u * g * row_bytes, 0, 0);
      f32x16 acc;
      const int row = 32 * rh + (lane & 31);
      const uint32_t a_row = buf * kTileBytes + (uint32_t)row * (kBW * 2);
      auto a_read = [&](int f) {
        const uint32_t chunk = (uint32_t)(2 * (f & 15) + (lane >> 5)) ^
                               (uint32_t)(row & 31);
        return *reinterpret_cast<lds_f32x4*>(
            lds3 + a_row + (f >> 4) * (kRows * kBW * 2) + 16u * chunk);
      };
      f32x4 a[4];
#pragma unroll
      for (int f = 0; f < 3; ++f) a[f] = a_read(f);
#pragma unroll
      for (int f = 0; f < 32; ++f) {
        if (f + 3 < 32) a[(f + 3) & 3] = a_read(f + 3);
        mfma_weight_frag(f, f == 0, a[f & 3], acc);
      }
      asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc));
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        // a lane: one channel, tokens 8 (e / 4) + 4 (lane / 32) + e % 4
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int t = 8 * (e >> 2) + (e & 3) + 4 * (lane >> 5);
          *reinterpret_cast<lds_f32*>(lds3 + patch +
                                      (t * kPatchFloats + (lane & 31)) * 4) =
              acc[8 * g + e];
        }
        float v[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const f32x4 r = *reinterpret_cast<lds_f32x4*>(
              lds3 + patch +
              ((lane >> 2) * kPatchFloats + 8 * (lane & 3) + 4 * q) * 4);
#pragma unroll
          for (int k = 0; k < 4; ++k) v[4 * q + k] = r[k];
        }
        asm volatile("" ::: "memory");  // (a wave's LDS instructions are in order)
        u32x4 out;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          out[k] = pack_bf16x2(
              v[2 * k] + __uint_as_float(old[g][k] << 16),
              v[2 * k + 1] + __uint_as_float(old[g][k] & 0xffff0000u));
        buffer_store_16(out, rdx, off + 16u * g * row_bytes, 0);
      }
    }
  }
}

// ---- column sums --------------------------------------------------------------
template <typename T>
struct Vec;
template <>
struct Vec<uint16_t> {
  static constexpr int n = 8;
  __device__ static void unpack(u32x4 r, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(r[i] << 16);
      v[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
  __device__ static u32x4 pack(float (&v)[8]) {
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    unpack(r, v);
    return r;
  }
};
template <>
struct Vec<float> {
  static constexpr int n = 4;
  __device__ static void unpack(u32x4 r, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(r[i]);
  }
  __device__ static u32x4 pack(float (&v)[4]) {
    return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]),
                 __float_as_uint(v[2]), __float_as_uint(v[3])};
  }
};

// Blocks of 256 threads: 32 lanes of 16 bytes along the columns, eight along
// the rows, eight rows each: 64 rows per block.
constexpr int kSumLanes = 32, kSumGroups = 8;
constexpr int kSumRows = kColSumRows / kSumGroups;

// This thread's sums of its rows -> the block's, in group order.
template <int N>
__device__ __forceinline__ void finish_col_sums(float (&sums)[N],
                                                float* partial, int W, int c,
                                                bool c_ok) {
  __shared__ float s[kSumGroups][kSumLanes * N + 4];
  const int l = threadIdx.x % kSumLanes, g = threadIdx.x / kSumLanes;
#pragma unroll
  for (int e = 0; e < N; ++e) s[g][l * N + e] = sums[e];
  __syncthreads();
  if (g == 0 && c_ok) {
#pragma unroll
    for (int e = 0; e < N; ++e) {
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < kSumGroups; ++k) v += s[k][l * N + e];
      partial[(int64_t)blockIdx.y * W + c + e] = v;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kSumLanes* kSumGroups)
col_sums_kernel(const T* __restrict__ in, float* __restrict__ partial, int64_t M,
                int W) {
  using V = Vec<T>;
  constexpr int N = V::n;
  const int c = ((int)blockIdx.x * kSumLanes + (int)threadIdx.x % kSumLanes) * N;
  const bool c_ok = c < W;
  const int64_t m0 = (int64_t)blockIdx.y * kColSumRows +
                     (threadIdx.x / kSumLanes) * kSumRows;
  u32x4 r[kSumRows];
#pragma unroll
  for (int i = 0; i < kSumRows; ++i)
    r[i] = c_ok && m0 + i < M
               ? *reinterpret_cast<const u32x4*>(in + (m0 + i) * W + c)
               : u32x4{0, 0, 0, 0};
  float sums[N];
#pragma unroll
  for (int e = 0; e < N; ++e) sums[e] = 0.0f;
#pragma unroll
  for (int i = 0; i < kSumRows; ++i) {
    float v[N];
    V::unpack(r[i], v);
#pragma unroll
    for (int e = 0; e < N; ++e) sums[e] += v[e];
  }
  finish_col_sums(sums, partial, W, c, c_ok);
}

template <typename T>
__global__ void __launch_bounds__(kSumLanes* kSumGroups)
gelu_mul_backward_sums_kernel(const T* __restrict__ dout,
                              const T* __restrict__ a, const T* __restrict__ g,
                              T* __restrict__ d_a, T* __restrict__ d_g,
                              float* __restrict__ partial, int64_t M, int W) {
  using V = Vec<T>;
  constexpr int N = V::n;
  const int c = ((int)blockIdx.x * kSumLanes + (int)threadIdx.x % kSumLanes) * N;
  const bool c_ok = c < W;
  const int64_t m0 = (int64_t)blockIdx.y * kColSumRows +
                     (threadIdx.x / kSumLanes) * kSumRows;
  u32x4 rd[kSumRows], ra[kSumRows], rg[kSumRows];
#pragma unroll
  for (int i = 0; i < kSumRows; ++i) {
    const int64_t at = c_ok && m0 + i < M ? (m0 + i) * W + c : 0;
    rd[i] = *reinterpret_cast<const u32x4*>(dout + at);
    ra[i] = *reinterpret_cast<const u32x4*>(a + at);
    rg[i] = *reinterpret_cast<const u32x4*>(g + at);
  }
  float sums[N];
#pragma unroll
  for (int e = 0; e < N; ++e) sums[e] = 0.0f;
#pragma unroll
  for (int i = 0; i < kSumRows; ++i) {
    float dv[N], av[N], gv[N], oa[N], og[N];
    V::unpack(rd[i], dv);
    V::unpack(ra[i], av);
    V::unpack(rg[i], gv);
#pragma unroll
    for (int e = 0; e < N; ++e)
      gelu_mul_backward_one<sizeof(T) == 2>(dv[e], av[e], gv[e], oa[e], og[e]);
    const u32x4 pa = V::pack(oa), pg = V::pack(og);  // (og: as stored)
    if (c_ok && m0 + i < M) {
      *reinterpret_cast<u32x4*>(d_a + (m0 + i) * W + c) = pa;
      *reinterpret_cast<u32x4*>(d_g + (m0 + i) * W + c) = pg;
#pragma unroll
      for (int e = 0; e < N; ++e) sums[e] += og[e];
    }
  }
  finish_col_sums(sums, partial, W, c, c_ok);
}

struct SumTasks {
  SumTask t[kMaxSumTasks];
  int first[kMaxSumTasks + 1];  // first block of each task
};
// A block: 64 columns, 16 rows at a time (a few hundred rows are all in flight
// after the second load of a thread).
constexpr int kSumWaves = 16;
template <typename T>
__global__ void __launch_bounds__(64 * kSumWaves) sum_rows_kernel(SumTasks p) {
  __shared__ float s[kSumWaves][64];
  int k = 0;
#pragma unroll
  for (int i = 1; i < kMaxSumTasks; ++i)
    if ((int)blockIdx.x >= p.first[i]) k = i;
  const SumTask t = p.t[k];
  const int n = ((int)blockIdx.x - p.first[k]) * 64 + (threadIdx.x & 63);
  const int g = threadIdx.x >> 6;
  float sum = 0.0f;
  if (n < t.n) {
#pragma unroll 8
    for (int r = g; r < t.rows; r += kSumWaves) sum += t.in[(int64_t)r * t.ld + n];
  }
  s[g][threadIdx.x & 63] = sum;
  __syncthreads();
  if (g == 0 && n < t.n) {
    const int l = threadIdx.x;
    float v = s[0][l];
#pragma unroll
    for (int k = 1; k < kSumWaves; ++k) v += s[k][l];
    store_scalar((T*)t.out + n, v);
  }
}

dim3 col_grid(int64_t M, int W, int per_lane) {
  return dim3((unsigned)((W / per_lane + kSumLanes - 1) / kSumLanes),
              (unsigned)((M + kColSumRows - 1) / kColSumRows));
}

}  // namespace

hipError_t launch_gates_dgrad(const void* dgx, const void* dga, const void* w_x,
                              const void* w_a, void* dx, int64_t M, int W, int H,
                              hipStream_t s) {
  if (M <= 0 || W != kBW * H || (int64_t)kRows * W * 2 >= (int64_t)0x7fffffff)
    return hipErrorInvalidValue;
  static OncePerDevice once;
  hipError_t e =
      set_max_dynamic_lds(once, (const void*)gates_dgrad_kernel, kDgradLds);
  if (e != hipSuccess) return e;
  const int64_t tiles = (M + kRows - 1) / kRows;
  int64_t ranges = 256 / H;  // one workgroup per CU
  if (ranges < 1) ranges = 1;
  if (ranges > tiles) ranges = tiles;
  gates_dgrad_kernel<<<dim3((unsigned)(ranges * H)), kThreads, kDgradLds, s>>>(
      (const uint16_t*)dgx, (const uint16_t*)dga, (const uint16_t*)w_x,
      (const uint16_t*)w_a, (uint16_t*)dx, M, W, H, (int)ranges);
  return hipGetLastError();
}

hipError_t launch_col_sums(const void* in, float* partial, int64_t M, int W,
                           int dtype, hipStream_t s) {
  const int per = dtype == 0 ? 4 : 8;
  if (M <= 0 || W % per || (M + kColSumRows - 1) / kColSumRows > 65535)
    return hipErrorInvalidValue;
  if (dtype == 0)
    col_sums_kernel<<<col_grid(M, W, per), kSumLanes * kSumGroups, 0, s>>>(
        (const float*)in, partial, M, W);
  else
    col_sums_kernel<<<col_grid(M, W, per), kSumLanes * kSumGroups, 0, s>>>(
        (const uint16_t*)in, partial, M, W);
  return hipGetLastError();
}

hipError_t launch_gelu_mul_backward_sums(const void* dout, const void* a,
                                         const void* g, void* d_a, void* d_g,
                                         float* partial, int64_t M, int W,
                                         int dtype, hipStream_t s) {
  const int per = dtype == 0 ? 4 : 8;
  if (M <= 0 || W % per || (M + kColSumRows - 1) / kColSumRows > 65535)
    return hipErrorInvalidValue;
  if (dtype == 0)
    gelu_mul_backward_sums_kernel<<<col_grid(M, W, per), kSumLanes * kSumGroups, 0,
                                    s>>>(
        (const float*)dout, (const float*)a, (const float*)g, (float*)d_a,
        (float*)d_g, partial, M, W);
  else
    gelu_mul_backward_sums_kernel<<<col_grid(M, W, per), kSumLanes * kSumGroups, 0,
                                    s>>>(
        (const uint16_t*)dout, (const uint16_t*)a, (const uint16_t*)g,
        (uint16_t*)d_a, (uint16_t*)d_g, partial, M, W);
  return hipGetLastError();
}

hipError_t launch_sum_rows(const SumTask* tasks, int count, int dtype,
                           hipStream_t s) {
  if (count < 1 || count > kMaxSumTasks) return hipErrorInvalidValue;
  SumTasks p{};
  int blocks = 0;
  for (int i = 0; i < kMaxSumTasks; ++i) {
    p.first[i] = blocks;
    if (i < count) {
      p.t[i] = tasks[i];
      blocks += (tasks[i].n + 63) / 64;
    } else {
      p.first[i] = 0x7fffffff;  // (never reached)
    }
  }
  if (blocks <= 0) return hipErrorInvalidValue;
  if (dtype == 0) sum_rows_kernel<float><<<dim3((unsigned)blocks), 64 * kSumWaves, 0, s>>>(p);
  else sum_rows_kernel<uint16_t><<<dim3((unsigned)blocks), 64 * kSumWaves, 0, s>>>(p);
  return hipGetLastError();
}

}  // namespace rg
