// One row of RMSNorm in bf16 and what its callers have around it: the pass of its own
// (rg_elementwise.hip) and the launch that has the layer behind it, too (rg_linear.hip).
#ifndef RG_NORM_ROW_H_
#define RG_NORM_ROW_H_

#include "rg_common.h"
#include "rg_internal.h"

namespace rg {

// The row a linear layer left as fp32 partial sums over slices of its K
// (rg_linear.hip): x = round(sum of the slices, in slice order, + bias).
struct PartialRows {
  const f32x4* sums;     // [slices][rows][width]
  int slices;
  int64_t slice_stride;  // rows * width / 4
  const u32x4* bias;     // [width] or null
};

// x / rms(x) * (1 + scale) of row `at`, every step rounded as written; 256 threads, t
// the thread's number.  One workgroup barrier, for which any other threads wait, too.
// SHARED: other workgroups of the launch read the row: agent-scope stores.
template <bool ADD, bool FROM_PARTIAL, bool SHARED>
__device__ __forceinline__ void rms_norm_row(
    const int t, const int64_t at, float* const partial, const u32x4* __restrict__ x,
    const PartialRows& part, const u32x4* __restrict__ addend,
    const u32x4* __restrict__ scale, u32x4* __restrict__ sum_out, u32x4* __restrict__ out,
    const int chunks, const float inv_width, const float eps) {
  const int64_t row = at * chunks;
  const u32x4* xr = x + row;
  u32x4* outr = out + row;
  u32x4 v[2];
  float sum = 0.0f;
  // A row of partial sums: everything is asked for before anything is used, in one
  // wait instead of one per slice and chunk (us replayed from a graph, where a launch
  // takes 2.5 whatever it does, three slices: 16 rows of 2560 4.05 / 3.68, of 4096
  // 4.81 / 3.77, 64 of 2560 5.78 / 4.08).  Lanes and slices beyond the last read the
  // last again.
  constexpr int kSlicesAhead = FROM_PARTIAL ? 3 : 1;
  f32x4 ahead[2][kSlicesAhead][2];
  u32x4 ahead_bias[2], ahead_addend[2], ahead_scale[2];
  if (FROM_PARTIAL) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int i = min(t + c * 256, chunks - 1);
#pragma unroll
      for (int k = 0; k < kSlicesAhead; ++k) {
        const f32x4* src =
            part.sums + (row + i) * 2 + min(k, part.slices - 1) * part.slice_stride;
        ahead[c][k][0] = src[0];
        ahead[c][k][1] = src[1];
      }
      if (ADD) ahead_addend[c] = addend[row + i];
      ahead_scale[c] = scale[i];
      // (where there is none, something else of the same size that is not used)
      ahead_bias[c] = (part.bias ? part.bias : scale)[i];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int i = t + c * 256;
    v[c] = u32x4{0u, 0u, 0u, 0u};
    if (!FROM_PARTIAL && i < chunks) v[c] = __builtin_nontemporal_load(xr + i);
    if (FROM_PARTIAL && i < chunks) {
      f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
      // (slices beyond the last add nothing)
#pragma unroll
      for (int k = 0; k < kSlicesAhead; ++k) {
        lo += k < part.slices ? ahead[c][k][0] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        hi += k < part.slices ? ahead[c][k][1] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      const f32x4* src = part.sums + (row + i) * 2;
      for (int k = kSlicesAhead; k < part.slices; ++k) {
        lo += src[k * part.slice_stride];
        hi += src[k * part.slice_stride + 1];
      }
      if (part.bias) {
        const u32x4 b = ahead_bias[c];
        lo += f32x4{__uint_as_float(b[0] << 16),
                    __uint_as_float(b[0] & 0xffff0000u),
                    __uint_as_float(b[1] << 16),
                    __uint_as_float(b[1] & 0xffff0000u)};
        hi += f32x4{__uint_as_float(b[2] << 16),
                    __uint_as_float(b[2] & 0xffff0000u),
                    __uint_as_float(b[3] << 16),
                    __uint_as_float(b[3] & 0xffff0000u)};
      }
      v[c] = u32x4{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]),
                   pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
      if (!ADD) sum_out[row + i] = v[c];
    }
    if (ADD && i < chunks) {
      const u32x4 w = FROM_PARTIAL ? ahead_addend[c]
                                   : __builtin_nontemporal_load(addend + row + i);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[c][k] = pack_bf16x2(
            __uint_as_float(v[c][k] << 16) + __uint_as_float(w[k] << 16),
            __uint_as_float(v[c][k] & 0xffff0000u) +
                __uint_as_float(w[k] & 0xffff0000u));
      sum_out[row + i] = v[c];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float lo = __uint_as_float(v[c][k] << 16);
      const float hi = __uint_as_float(v[c][k] & 0xffff0000u);
      sum += round_to_bf16(lo * lo);
      sum += round_to_bf16(hi * hi);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if ((t & 63) == 0) partial[t >> 6] = sum;
  __syncthreads();
  sum = (partial[0] + partial[1]) + (partial[2] + partial[3]);
  const float var = round_to_bf16(sum * inv_width);
  const float r = round_to_bf16(1.0f / sqrtf(round_to_bf16(var + eps)));
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int i = t + c * 256;
    if (i >= chunks) continue;
    const u32x4 g = FROM_PARTIAL ? ahead_scale[c] : scale[i];
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float lo = round_to_bf16(__uint_as_float(v[c][k] << 16) * r) *
                       round_to_bf16(__uint_as_float(g[k] << 16) + 1.0f);
      const float hi =
          round_to_bf16(__uint_as_float(v[c][k] & 0xffff0000u) * r) *
          round_to_bf16(__uint_as_float(g[k] & 0xffff0000u) + 1.0f);
      o[k] = pack_bf16x2(lo, hi);
    }
    if (SHARED) {
      uint64_t* const to = reinterpret_cast<uint64_t*>(outr + i);
#pragma unroll
      for (int k = 0; k < 2; ++k)
        __hip_atomic_store(to + k, (uint64_t)o[2 * k + 1] << 32 | o[2 * k],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      __builtin_nontemporal_store(o, outr + i);
    }
  }
}

}  // namespace rg
#endif  // RG_NORM_ROW_H_
