// Prompt-pass attention of the local-attention block: sliding-window,
// multi-query (all heads share one key/value head), causal within a document
// (recurrentgemma/torch/modules.py:404-476 with the mask of :86-127), bf16,
// head dimension 256, as one kernel -- scores, mask, softmax and the weighted
// sum of the values without the [T, T] matrices in memory.
//
// The mask of a prompt is a band: query t sees the keys lo[t] .. t, where
// lo[t] = max(first token of t's document, t - window) is supplied by the
// caller (non-decreasing in t).
//
// One workgroup of four waves per (row, head, 128 queries); a wave owns 32
// queries.  Keys and values come by in tiles of 64 keys, staged in LDS for the
// four waves.  Both products are v_mfma_f32_32x32x16_bf16 with the QUERIES as
// the 32 columns of the result:
//   S^T [32 keys x 32 queries]  = K tile [32 x 256]   x Q^T [256 x 32]
//   O^T [256 x 32 queries]     += V^T tile [256 x 32] x P^T [32 keys x 32]
// so a lane (query l % 32, half l / 32) holds, of every result, one query's
// values: the softmax statistics of a query are per-lane scalars (one exchange
// between the two halves per tile), the 16 scores a lane holds become, as they
// lie, its operand of the second product, and rescaling O is a multiplication
// by a per-lane scalar.  Which keys sit in which contraction slot of the second
// product is free as long as both operands agree: the S^T result gives half h
// of a lane the keys 8 j + 4 h + i (j = 0..3, i = 0..3), so the values are laid
// out in LDS in that order.  The values arrive transposed ([row, 256, T]: the
// caller's one extra pass over them), which makes the contraction index the
// contiguous one of both operands of both products.
//
// What a block does around that for a prompt -- rotary embedding, the values'
// transposition, the ring cache it leaves -- is attn_prompt_prepare_kernel at
// the end of this file; the queries take their rotary embedding inside the
// attention kernel.
#include <utility>

#include "rg_common.h"
#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kAttnHd = 256;
constexpr int kAttnQ = 128;  // queries per workgroup
constexpr int kAttnK = 64;   // keys per tile
constexpr int kAttnKB = kAttnK / 32;  // blocks of 32 keys (one S^T result each)
constexpr int kAttnChunks = kAttnK * 32 / 256;  // 16-byte chunks per thread, tile and tensor
// K tile rows (one key, 512 B) padded to 528 B, V^T tile rows (one of the 256
// dimensions, 64 keys = 128 B) to 144 B: the 16-byte operand reads of 16
// consecutive rows fall on distinct banks.
constexpr int kKRowBytes = 528;
constexpr int kVRowBytes = 2 * kAttnK + 16;
constexpr int kKTileBytes = kAttnK * kKRowBytes;
constexpr int kVTileBytes = kAttnHd * kVRowBytes;

union AFrag {
  bf16x8 v;
  f32x4 q;
  uint32_t u[4];
};

// The 128 output accumulators of a lane (O^T: 8 blocks of 32 dimensions, 16
// registers each) live in the accumulation registers a[0:127] for the whole
// kernel, written and read by inline assembly with the register numbers
// spelled out: the second product accumulates into them tile after tile, and
// nothing else touches them but the rare rescaling and the final store (left
// to the register allocator they were moved between the two register files
// every tile, 256 moves for 32 matrix instructions).  The build checks that
// the compiler allocates no accumulation register of its own in this file.
#define RG_ATTN_LAST_AGPR "a127"

template <int N>
__device__ __forceinline__ float acc_read() {
  float t;
  asm volatile("v_accvgpr_read_b32 %0, a[%c1]" : "=v"(t) : "n"(N));
  return t;
}
template <int N>
__device__ __forceinline__ void acc_write(float t) {
  asm volatile("v_accvgpr_write_b32 a[%c1], %0" ::"v"(t), "n"(N)
               : RG_ATTN_LAST_AGPR);
}
template <int... I>
__device__ __forceinline__ void acc_fill(float v,
                                         std::integer_sequence<int, I...>) {
  (acc_write<I>(v), ...);
}
template <int... I>
__device__ __forceinline__ void acc_scale(float f,
                                          std::integer_sequence<int, I...>) {
  (acc_write<I>(acc_read<I>() * f), ...);
}
// block BLK of O^T += a x b
template <int BLK>
__device__ __forceinline__ void acc_mfma(const f32x4& a, const f32x4& b) {
  asm volatile(
      "v_mfma_f32_32x32x16_bf16 a[%c2:%c2+15], %0, %1, a[%c2:%c2+15]" ::"v"(a),
      "v"(b), "n"(16 * BLK)
      : RG_ATTN_LAST_AGPR);
}
// The compiler does not count the wait states between a matrix instruction in
// inline assembly and a read of its result.
__device__ __forceinline__ void wait_for_matrix_results() {
  asm volatile("s_nop 15\n\ts_nop 7");
}

// Rotary embedding of the first half of a query's dimensions (elements i and
// i + 64, i < 64) where the query lies as operand fragments: k-steps 0..3 hold
// this lane's elements 16 ks + 8 half + 0..7, k-steps 4..7 their partners.
// `table` is the query's row of sines and cosines (see
// attn_prompt_prepare_kernel).  The arithmetic of rg_rope_pair, element for
// element: products and sums rounded one by one.
__device__ __forceinline__ void rotate_query(AFrag (&qf)[16],
                                             const u32x4 (&table)[8]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      float vlo[2], vhi[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t sc = table[2 * ks + (w >> 1)][2 * (w & 1) + e];
        const float sn = __uint_as_float(sc << 16);
        const float cs = __uint_as_float(sc & 0xffff0000u);
        const uint32_t l = qf[ks].u[w], h = qf[ks + 4].u[w];
        const float lo = __uint_as_float(e == 0 ? l << 16 : l & 0xffff0000u);
        const float hi = __uint_as_float(e == 0 ? h << 16 : h & 0xffff0000u);
        vlo[e] = round_to_bf16(lo * cs) - round_to_bf16(hi * sn);
        vhi[e] = round_to_bf16(hi * cs) + round_to_bf16(lo * sn);
      }
      qf[ks].u[w] = pack_bf16x2(vlo[0], vlo[1]);
      qf[ks + 4].u[w] = pack_bf16x2(vhi[0], vhi[1]);
    }
  }
}

// ROPE: the queries come before their rotary embedding and take it here, in
// the registers they are loaded to (p.rope_table); a pass of its own over them
// reads and writes every query once more (8 x 2047 tokens, 10 heads: 43 us).
template <bool ROPE>
__global__ void __launch_bounds__(256)
attn_prefill_bf16_kernel(AttnPrefillArgs p) {
  extern __shared__ __align__(16) unsigned char attn_lds[];
  unsigned char* const k_tile = attn_lds;                    // two buffers
  unsigned char* const v_tile = attn_lds + 2 * kKTileBytes;  // two buffers

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, half = lane >> 5;
  const int qtiles = (p.T + kAttnQ - 1) / kAttnQ;
  // Workgroups go to the eight XCDs in turn (linear id modulo 8), each with an
  // L2 of its own: the ids are dealt out so that one XCD gets a contiguous run
  // of (row, head, query tile) triples, i.e. a row's keys and values are
  // pulled through one L2 instead of all eight.
  unsigned id = blockIdx.x;
  {
    const unsigned per_xcd = gridDim.x / 8;
    if (id < 8 * per_xcd) id = (id & 7) * per_xcd + (id >> 3);
  }
  // the longest workgroups (last query tiles) first
  const int qt = qtiles - 1 - (int)(id % qtiles);
  const int head = (int)(id / qtiles) % p.H;
  const int b = (int)(id / qtiles) / p.H;
  const int T = p.T;
  const int q0 = qt * kAttnQ;
  const int qw0 = q0 + 32 * wave;  // this wave's first query
  const int q = qw0 + n;           // this lane's query

  // descriptors over this row's tensors
  const uint32_t q_row_bytes = (uint32_t)p.H * kAttnHd * 2u;
  const __amdgpu_buffer_rsrc_t rq =
      make_rsrc((const char*)p.q + (int64_t)b * T * q_row_bytes,
                (uint32_t)T * q_row_bytes);
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(
      (char*)p.out + (int64_t)b * T * q_row_bytes, (uint32_t)T * q_row_bytes);
  const __amdgpu_buffer_rsrc_t rk =
      make_rsrc((const char*)p.k + (int64_t)b * T * (kAttnHd * 2),
                (uint32_t)T * (kAttnHd * 2u));
  const uint32_t vt_row_bytes = (uint32_t)p.T_pad * 2u;
  const __amdgpu_buffer_rsrc_t rv =
      make_rsrc((const char*)p.v_t + (int64_t)b * kAttnHd * vt_row_bytes,
                (uint32_t)kAttnHd * vt_row_bytes);
  const __amdgpu_buffer_rsrc_t rlo = make_rsrc(
      (const char*)p.lo + (int64_t)b * T * 4, (uint32_t)T * 4u);

  // first visible key of this lane's query, and of the tile's / wave's first
  // query (lo is non-decreasing: they bound the keys the tile / wave needs)
  auto lo_at = [&](int t) {
    return (int)__builtin_amdgcn_raw_buffer_load_b32(
        rlo, t < T ? (uint32_t)t * 4u : kBufferOutOfRange, 0, 0);
  };
  const int lo_q = q < T ? lo_at(q) : 0x7fffffff;
  const int lo_tile = __builtin_amdgcn_readfirstlane(lo_at(q0));
  const int lo_wave =
      __builtin_amdgcn_readfirstlane(qw0 < T ? lo_at(qw0) : 0x7fffffff);
  const int q_last_tile = q0 + kAttnQ - 1 < T - 1 ? q0 + kAttnQ - 1 : T - 1;
  const int q_last_wave = qw0 + 31 < T - 1 ? qw0 + 31 : T - 1;
  const int kt_begin = lo_tile / kAttnK;
  const int kt_end = q_last_tile / kAttnK;  // inclusive

  // (after the bounds, which the first tile's addresses wait for: loads return
  // in order, and the tile is requested with the queries on their way)
  // this lane's query as the B operand of the first product: 16 k-steps of
  // 8 dimensions (16 bytes); queries past the end read as zero
  AFrag qf[16];
  {
    const uint32_t off = (uint32_t)q * q_row_bytes + (uint32_t)head * 512u +
                         16u * (uint32_t)half;
#pragma unroll
    for (int ks = 0; ks < 16; ++ks)
      qf[ks].q = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     rq, q < T ? off + 32u * ks : kBufferOutOfRange, 0, 0));
  }
  u32x4 table[ROPE ? 8 : 1];  // this lane's share of the query's sines, cosines
  if (ROPE) {
    const __amdgpu_buffer_rsrc_t rt =
        make_rsrc((const char*)p.rope_table + (int64_t)b * T * 256,
                  (uint32_t)T * 256u);
    const uint32_t off = (uint32_t)q * 256u + 32u * (uint32_t)half;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      table[i] = __builtin_amdgcn_raw_buffer_load_b128(
          rt, q < T ? off + 64u * (i >> 1) + 16u * (i & 1) : kBufferOutOfRange,
          0, 0);
  }

  acc_fill(0.0f, std::make_integer_sequence<int, 128>{});
  float m_run = -__builtin_inff();  // running maximum, in units of log2
  float l_run = 0.0f;               // running sum over this half's keys
  const float scale_log2 = p.scale * kLog2e;

  // staging: 16-byte chunks, kAttnChunks per thread, tile and tensor; the
  // chunks of tile kt + 1 are requested as soon as tile kt is in LDS and
  // arrive while it is worked on
  u32x4 kc[kAttnChunks], vc[kAttnChunks];
  auto request_tile = [&](int kt) {
    const int key0 = kt * kAttnK;
#pragma unroll
    for (int i = 0; i < kAttnChunks; ++i) {
      const int c = tid + 256 * i;
      const int krow = c >> 5, kcol = c & 31;
      const int key = key0 + krow;
      kc[i] = __builtin_amdgcn_raw_buffer_load_b128(
          rk, key < T ? (uint32_t)key * 512u + 16u * kcol : kBufferOutOfRange,
          0, 0);
      const int d = c / (kAttnK / 8), part = c % (kAttnK / 8);
      vc[i] = __builtin_amdgcn_raw_buffer_load_b128(
          rv, (uint32_t)d * vt_row_bytes + (uint32_t)(key0 + 8 * part) * 2u, 0,
          0);
    }
  };
  auto stage_tile = [&](int buf) {
    unsigned char* const kt_ = k_tile + buf * kKTileBytes;
    unsigned char* const vt_ = v_tile + buf * kVTileBytes;
#pragma unroll
    for (int i = 0; i < kAttnChunks; ++i) {
      const int c = tid + 256 * i;
      const int krow = c >> 5, kcol = c & 31;
      *reinterpret_cast<u32x4*>(kt_ + krow * kKRowBytes + 16 * kcol) = kc[i];
      const int d = c / (kAttnK / 8), part = c % (kAttnK / 8);
      // keys 8 part .. 8 part + 7 of the tile: group s = part / 2 of 16 keys,
      // stored as [keys 0-3, 8-11 | keys 4-7, 12-15] of the group
      unsigned char* const vb =
          vt_ + d * kVRowBytes + 32 * (part >> 1) + 8 * (part & 1);
      *reinterpret_cast<u32x2*>(vb) = u32x2{vc[i][0], vc[i][1]};
      *reinterpret_cast<u32x2*>(vb + 16) = u32x2{vc[i][2], vc[i][3]};
    }
  };
  // Two LDS buffers: while tile kt is worked on out of one, tile kt + 1
  // arrives in registers and is written to the other afterwards; one barrier
  // per tile.
  request_tile(kt_begin);
  if constexpr (ROPE) rotate_query(qf, table);
  stage_tile(0);
  __syncthreads();
  if (kt_begin < kt_end) request_tile(kt_begin + 1);
  // last query of this wave sees from lo_last_wave on (lo is non-decreasing)
  const int lo_last_wave = __builtin_amdgcn_readfirstlane(lo_at(q_last_wave));
  for (int kt = kt_begin; kt <= kt_end; ++kt) {
    const int key0 = kt * kAttnK;
    const int buf = (kt - kt_begin) & 1;
    const unsigned char* const kt_ = k_tile + buf * kKTileBytes;
    const unsigned char* const vt_ = v_tile + buf * kVTileBytes;

    // tiles outside what this wave's queries can see are skipped (wave-uniform)
    if (!(key0 > q_last_wave || key0 + kAttnK - 1 < lo_wave)) {
      // ---- S^T = K tile x Q^T ----------------------------------------------
      // (inline assembly with the results in ordinary registers: a matrix
      // builtin lets the compiler pick accumulation registers for the result,
      // and it picks a[0:15].  The compiler moves no LDS read across such a
      // statement, so the operands are requested by hand, four fragments
      // ahead of the instructions that use them.)
      f32x16 s[kAttnKB];
      {
        constexpr int kFrags = 16 * kAttnKB, kBatch = 4;
        auto k_frag = [&](int f) {  // fragment f: k-step f / KB, key block f % KB
          return *reinterpret_cast<const f32x4*>(
              kt_ + (32 * (f % kAttnKB) + n) * kKRowBytes + 32 * (f / kAttnKB) +
              16 * half);
        };
        f32x4 fr[2][kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; ++i) fr[0][i] = k_frag(i);
#pragma unroll
        for (int bt = 0; bt < kFrags / kBatch; ++bt) {
          if (bt + 1 < kFrags / kBatch) {
#pragma unroll
            for (int i = 0; i < kBatch; ++i)
              fr[(bt + 1) & 1][i] = k_frag((bt + 1) * kBatch + i);
          }
#pragma unroll
          for (int i = 0; i < kBatch; ++i) {
            const int f = bt * kBatch + i;
            const int ks = f / kAttnKB, kb = f % kAttnKB;
            if (ks == 0)
              asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0"
                           : "=&v"(s[kb])
                           : "v"(fr[bt & 1][i]), "v"(qf[ks].q));
            else
              asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
                           : "+v"(s[kb])
                           : "v"(fr[bt & 1][i]), "v"(qf[ks].q));
          }
        }
      }
      // (tied to the scores: nothing that reads them may be scheduled above
      // the wait)
#pragma unroll
      for (int kb = 0; kb < kAttnKB; ++kb) asm volatile("" : "+v"(s[kb]));
      wait_for_matrix_results();
#pragma unroll
      for (int kb = 0; kb < kAttnKB; ++kb) asm volatile("" : "+v"(s[kb]));
      // ---- mask (only where the band's edges cross the tile) ----------------
      const bool interior = key0 + kAttnK - 1 <= qw0 && key0 >= lo_last_wave;
      if (!interior) {
#pragma unroll
        for (int kb = 0; kb < kAttnKB; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = key0 + 32 * kb + 8 * (r >> 2) + 4 * half + (r & 3);
            s[kb][r] = (key >= lo_q && key <= q) ? s[kb][r] : -__builtin_inff();
          }
      }
      // ---- running maximum (in units of log2), moved only when the tile's
      //      exceeds it by more than 2^8: the accumulators are rescaled rarely --
      float tile_max = s[0][0];
#pragma unroll
      for (int kb = 0; kb < kAttnKB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s[kb][r]);
      {
        const auto sw = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(tile_max), __float_as_uint(tile_max), false, false);
        tile_max = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      tile_max *= scale_log2;  // (the scale is positive)
      if (__ballot(tile_max > m_run + 8.0f) != 0) {
        const float m_new = fmaxf(m_run, tile_max);
        // (no visible key so far: keep every exponent finite)
        const float alpha = __builtin_amdgcn_exp2f(
            m_run - (m_new == -__builtin_inff() ? 0.0f : m_new));
        // (before a query's first visible key its accumulators are zeros)
        const bool started = __ballot(m_run != -__builtin_inff()) != 0;
        m_run = m_new;
        l_run *= alpha;
        if (started) {
          wait_for_matrix_results();
          acc_scale(alpha, std::make_integer_sequence<int, 128>{});
        }
      }
      const float m_sub = m_run == -__builtin_inff() ? 0.0f : m_run;
      AFrag pf[2 * kAttnKB];
#pragma unroll
      for (int kb = 0; kb < kAttnKB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float p0 = __builtin_amdgcn_exp2f(
              __builtin_fmaf(s[kb][r], scale_log2, -m_sub));
          const float p1 = __builtin_amdgcn_exp2f(
              __builtin_fmaf(s[kb][r + 1], scale_log2, -m_sub));
          l_run += p0 + p1;
          pf[2 * kb + (r >> 3)].u[(r & 7) >> 1] = pack_bf16x2(p0, p1);
        }
      // ---- O^T += V^T tile x P^T: the eight blocks of a 16-key step one after
      //      the other (independent accumulators), the operands of the next
      //      step requested before ------------------------------------------------
      {
        auto v_frag = [&](int ss, int blk) {
          return *reinterpret_cast<const f32x4*>(
              vt_ + (32 * blk + n) * kVRowBytes + 32 * ss + 16 * half);
        };
        // batch bt: 16-key step bt / 2, blocks 4 (bt % 2) .. + 3
        f32x4 fr[2][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) fr[0][i] = v_frag(0, i);
#pragma unroll
        for (int bt = 0; bt < 4 * kAttnKB; ++bt) {
          if (bt + 1 < 4 * kAttnKB) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              fr[(bt + 1) & 1][i] = v_frag((bt + 1) >> 1, 4 * ((bt + 1) & 1) + i);
          }
          const f32x4& pq = pf[bt >> 1].q;
          if (bt & 1) {
            acc_mfma<4>(fr[bt & 1][0], pq);
            acc_mfma<5>(fr[bt & 1][1], pq);
            acc_mfma<6>(fr[bt & 1][2], pq);
            acc_mfma<7>(fr[bt & 1][3], pq);
          } else {
            acc_mfma<0>(fr[bt & 1][0], pq);
            acc_mfma<1>(fr[bt & 1][1], pq);
            acc_mfma<2>(fr[bt & 1][2], pq);
            acc_mfma<3>(fr[bt & 1][3], pq);
          }
        }
      }
    }
    if (kt < kt_end) {
      stage_tile(buf ^ 1);  // tile kt + 1; that buffer's readers passed the
      __syncthreads();      // barrier of the previous round
      if (kt + 1 < kt_end) request_tile(kt + 2);
    }
  }

  // ---- normalise and store: this lane's query, dimensions
  //      32 blk + 8 j + 4 half + i ---------------------------------------------
  wait_for_matrix_results();
  float l_total;
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(l_run), __float_as_uint(l_run), false, false);
    l_total = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  const float inv = l_total > 0.0f ? 1.0f / l_total : 0.0f;
  const uint32_t out_off = (uint32_t)q * q_row_bytes + (uint32_t)head * 512u;
  auto store4 = [&](int d0, float o0, float o1, float o2, float o3) {
    __builtin_amdgcn_raw_buffer_store_b64(
        u32x2{pack_bf16x2(o0 * inv, o1 * inv), pack_bf16x2(o2 * inv, o3 * inv)},
        ro, q < T ? out_off + (uint32_t)(d0 + 4 * half) * 2u : kBufferOutOfRange,
        0, 0);
  };
#define RG_ATTN_STORE(BLK, J)                                              \
  store4(32 * BLK + 8 * J, acc_read<16 * BLK + 4 * J>(),                   \
         acc_read<16 * BLK + 4 * J + 1>(), acc_read<16 * BLK + 4 * J + 2>(), \
         acc_read<16 * BLK + 4 * J + 3>());
#define RG_ATTN_STORE_BLK(BLK) \
  RG_ATTN_STORE(BLK, 0) RG_ATTN_STORE(BLK, 1) RG_ATTN_STORE(BLK, 2) RG_ATTN_STORE(BLK, 3)
  RG_ATTN_STORE_BLK(0) RG_ATTN_STORE_BLK(1) RG_ATTN_STORE_BLK(2) RG_ATTN_STORE_BLK(3)
  RG_ATTN_STORE_BLK(4) RG_ATTN_STORE_BLK(5) RG_ATTN_STORE_BLK(6) RG_ATTN_STORE_BLK(7)
#undef RG_ATTN_STORE_BLK
#undef RG_ATTN_STORE
}

// ---------------------------------------------------------------- prepare --
// Everything of the block between its projections and the attention kernel,
// in one pass over the keys and values (recurrentgemma/torch/modules.py:431-440
// and the ring cache of a prompt, :253-283): rotary embedding of the keys, the
// sines and cosines the queries are rotated with (one word per token and pair:
// sine in the low half, cosine in the high half, bf16), the values transposed
// for the second product (zeros behind the last token), the last min(window, T)
// keys and values in their ring slots, zeros in the slots never written, and
// the token count.
//
// One workgroup per (row, 32 tokens and 32 ring slots), which leaves the chip
// full from 8 x 1024 tokens on.  Bound by memory (8 x 2047 tokens: 17 MB in,
// 38 MB out); the tensor operations it replaces were ten launches, 146 us
// there.  32 tokens make runs of 64 bytes of a transposed row; with 64 a single
// prompt fills half as many CUs.
constexpr int kPrepTokens = 32;
constexpr int kPrepStride = kAttnHd + 8;  // of a token's values in LDS

__device__ __forceinline__ int64_t position_at(const AttnPromptArgs& p,
                                               int64_t i) {
  return p.pos_kind == kSegI64
             ? reinterpret_cast<const int64_t*>(p.pos)[i]
             : (int64_t)reinterpret_cast<const int32_t*>(p.pos)[i];
}

__global__ void __launch_bounds__(256)
attn_prompt_prepare_kernel(AttnPromptArgs p) {
#pragma clang fp contract(off)
  __shared__ __align__(16) uint16_t values[kPrepTokens * kPrepStride];
  const int tid = threadIdx.x;
  const int T = p.T, b = (int)(blockIdx.x / p.groups);
  const int t0 = (int)(blockIdx.x % p.groups) * kPrepTokens;
  const int64_t row0 = (int64_t)b * T;
  const uint16_t* const k = p.k + row0 * kAttnHd;
  const uint16_t* const v = p.v + row0 * kAttnHd;
  uint16_t* const k_out = p.k_rot + row0 * kAttnHd;
  const bool cache = p.ring_k != nullptr;
  uint16_t* const ring_k = p.ring_k + (int64_t)b * p.window * kAttnHd;
  uint16_t* const ring_v = p.ring_v + (int64_t)b * p.window * kAttnHd;

  // token t of the last `kept` lies in slot (t - (T - kept) + shift) % kept
  const int kept = p.window < T ? p.window : T;
  int shift = 0;
  if (cache) {
    const int count = (int)position_at(p, row0 + T - 1) + 1;
    shift = count % p.window;
    if (shift < 0) shift += p.window;
    if (t0 == 0 && tid == 0) p.num_tokens[b] = count;
  }
  auto slot_of = [&](int t) {  // -1: not kept
    const int i = t - (T - kept);
    return cache && i >= 0 ? (int)(((int64_t)i + shift) % kept) : -1;
  };

  // keys, rotated half: thread = 8 pairs of one token
  const int t_of = t0 + tid / 8;
  if (t_of < T) {
    const int i0 = 8 * (tid % 8);
    const u32x4 lo4 =
        *reinterpret_cast<const u32x4*>(k + (int64_t)t_of * kAttnHd + i0);
    const u32x4 hi4 =
        *reinterpret_cast<const u32x4*>(k + (int64_t)t_of * kAttnHd + 64 + i0);
    const float at = p.pos_kind == kSegI64
                         ? (float)position_at(p, row0 + t_of)
                         : (float)(int32_t)position_at(p, row0 + t_of);
    u32x4 olo, ohi, table[2];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      float vlo[2], vhi[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float angle = at * p.inv_freq[i0 + 2 * w + e];
        const float sn = round_to_bf16(sinf(angle));
        const float cs = round_to_bf16(cosf(angle));
        table[w >> 1][2 * (w & 1) + e] =
            (__float_as_uint(sn) >> 16) | (__float_as_uint(cs) & 0xffff0000u);
        const float lo =
            __uint_as_float(e == 0 ? lo4[w] << 16 : lo4[w] & 0xffff0000u);
        const float hi =
            __uint_as_float(e == 0 ? hi4[w] << 16 : hi4[w] & 0xffff0000u);
        vlo[e] = round_to_bf16(lo * cs) - round_to_bf16(hi * sn);
        vhi[e] = round_to_bf16(hi * cs) + round_to_bf16(lo * sn);
      }
      olo[w] = pack_bf16x2(vlo[0], vlo[1]);
      ohi[w] = pack_bf16x2(vhi[0], vhi[1]);
    }
    u32x4* const tab =
        reinterpret_cast<u32x4*>(p.rope_table + (row0 + t_of) * 64 + i0);
    tab[0] = table[0];
    tab[1] = table[1];
    uint16_t* const dst = k_out + (int64_t)t_of * kAttnHd + i0;
    *reinterpret_cast<u32x4*>(dst) = olo;
    *reinterpret_cast<u32x4*>(dst + 64) = ohi;
    const int slot = slot_of(t_of);
    if (slot >= 0) {
      uint16_t* const r = ring_k + (int64_t)slot * kAttnHd + i0;
      *reinterpret_cast<u32x4*>(r) = olo;
      *reinterpret_cast<u32x4*>(r + 64) = ohi;
    }
  }
  // keys, the half that is not rotated
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int t = t0 + 16 * j + tid / 16;
    const int d = 128 + 8 * (tid % 16);
    if (t < T) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(k + (int64_t)t * kAttnHd + d);
      *reinterpret_cast<u32x4*>(k_out + (int64_t)t * kAttnHd + d) = w;
      const int slot = slot_of(t);
      if (slot >= 0)
        *reinterpret_cast<u32x4*>(ring_k + (int64_t)slot * kAttnHd + d) = w;
    }
  }
  // values: to their ring slots, and through LDS into transposed rows
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = 8 * j + tid / 32, t = t0 + i;
    const int d = 8 * (tid % 32);
    u32x4 w = {0, 0, 0, 0};
    if (t < T) {
      w = *reinterpret_cast<const u32x4*>(v + (int64_t)t * kAttnHd + d);
      const int slot = slot_of(t);
      if (slot >= 0)
        *reinterpret_cast<u32x4*>(ring_v + (int64_t)slot * kAttnHd + d) = w;
    }
    *reinterpret_cast<u32x4*>(values + i * kPrepStride + d) = w;
  }
  // ring slots that no token of the prompt fills
  if (cache) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int slot = t0 + 8 * j + tid / 32;
      if (slot >= kept && slot < p.window) {
        const int64_t at = (int64_t)slot * kAttnHd + 8 * (tid % 32);
        *reinterpret_cast<u32x4*>(ring_k + at) = u32x4{0, 0, 0, 0};
        *reinterpret_cast<u32x4*>(ring_v + at) = u32x4{0, 0, 0, 0};
      }
    }
  }
  __syncthreads();
  if (t0 < p.T_pad) {  // (T_pad is a multiple of 64: all 32 columns exist)
    uint16_t* const vt = p.v_t + (int64_t)b * kAttnHd * p.T_pad + t0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 64 * j + tid / 4, part = tid % 4;
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint16_t* const c =
            values + (8 * part + 2 * e) * kPrepStride + d;
        w[e] = (uint32_t)c[0] | ((uint32_t)c[kPrepStride] << 16);
      }
      *reinterpret_cast<u32x4*>(vt + (int64_t)d * p.T_pad + 8 * part) = w;
    }
  }
}

// First key that each query of a prompt sees: the later of the start of its
// document (the last position 0 at or before it, else the row's first token)
// and the token `window` before it.  One workgroup per row, 1024 tokens at a
// time; within a wave the last start is the highest set bit of a ballot.
__global__ void __launch_bounds__(1024)
first_key_kernel(const void* pos, int pos_kind, int32_t* __restrict__ first,
                 int T, int window) {
  __shared__ int last[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row0 = (int64_t)blockIdx.x * T;
  int carry = 0;  // start of the document that reaches into this round
  for (int t0 = 0, round = 0; t0 < T; t0 += 1024, ++round) {
    const int t = t0 + tid;
    bool starts = false;
    if (t < T)
      starts = pos_kind == kSegI64
                   ? reinterpret_cast<const int64_t*>(pos)[row0 + t] == 0
                   : reinterpret_cast<const int32_t*>(pos)[row0 + t] == 0;
    const uint64_t mask = __ballot(starts);
    int* const found = last[round & 1];
    if (lane == 0)
      found[wave] = mask ? t0 + 64 * wave + 63 - __builtin_clzll(mask) : -1;
    __syncthreads();
    const uint64_t upto = mask & (~(uint64_t)0 >> (63 - lane));
    int start = upto ? t0 + 64 * wave + 63 - __builtin_clzll(upto) : -1;
    int before = carry;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) before = max(before, found[w]);
      carry = max(carry, found[w]);
    }
    start = max(start, before);
    if (t < T) first[row0 + t] = max(start, t - window);
  }
}

}  // namespace

hipError_t launch_attn_prompt_prepare(const AttnPromptArgs& args,
                                      hipStream_t s) {
  AttnPromptArgs a = args;
  const int64_t tokens = a.ring_k && a.window > a.T_pad ? a.window : a.T_pad;
  const int64_t groups = (tokens + kPrepTokens - 1) / kPrepTokens;
  if (groups <= 0 || a.B <= 0 || groups * a.B > 0x7fffffff)
    return hipErrorInvalidValue;
  a.groups = (unsigned)groups;
  attn_prompt_prepare_kernel<<<dim3((unsigned)(groups * a.B)), 256, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_first_key(const void* pos, int pos_kind, int32_t* first,
                            int B, int T, int window, hipStream_t s) {
  first_key_kernel<<<dim3((unsigned)B), 1024, 0, s>>>(pos, pos_kind, first, T,
                                                      window);
  return hipGetLastError();
}

hipError_t launch_attn_prefill_bf16(const AttnPrefillArgs& a, hipStream_t s) {
  // needs head dimension 256, T_pad a multiple of 64 >= T, and rows whose byte
  // offsets fit 32 bits (checked by the caller)
  const int64_t qtiles = (a.T + kAttnQ - 1) / kAttnQ;
  const int64_t blocks = qtiles * a.H * a.B;
  if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
  constexpr size_t lds = 2 * (size_t)(kKTileBytes + kVTileBytes);
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  static OncePerDevice once[2];
  const bool rope = a.rope_table != nullptr;
  hipError_t e = set_max_dynamic_lds(
      once[rope], rope ? (const void*)attn_prefill_bf16_kernel<true>
                       : (const void*)attn_prefill_bf16_kernel<false>, lds);
  if (e != hipSuccess) return e;
  if (rope)
    attn_prefill_bf16_kernel<true><<<dim3((unsigned)blocks), 256, lds, s>>>(a);
  else
    attn_prefill_bf16_kernel<false><<<dim3((unsigned)blocks), 256, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace rg
