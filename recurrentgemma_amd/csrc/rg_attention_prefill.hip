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
// A wave owns 48 queries of one head (32 in short prompts), a workgroup four such waves: heads of the same queries first, since all heads read the same keys and
// values.  They come by in blocks of 32 keys, global -> LDS by the memory pipe, three
// blocks ahead (a ring of four each), one barrier per block.  Both products are
// v_mfma_f32_16x16x32_bf16 with the QUERIES as the 16 columns of the result:
//   S^T [16 keys x 16 queries]  = K [16 x 256]     x Q^T [256 x 16]
//   O^T [16 dims x 16 queries] += V^T [16 x 32 keys] x P^T [32 keys x 16]
// so a lane (query l % 16, quarter l / 16) holds, of every result, one query's values:
// the softmax statistics of a query are per-lane scalars, the 8 scores a lane holds of
// a query become, as they lie, its operand of the second product, and rescaling O is a
// multiplication by a per-lane scalar.  Which keys sit in which contraction slot of the
// second product is free as long as both operands agree: the S^T results give quarter g
// the keys 4 g + i and 16 + 4 g + i (i = 0..3), and so the values are read from LDS, by
// ds_read_b64_tr_b16 where they lie key by key.
//
// One wave per SIMD, so what it overlaps it overlaps by its own order: the scores of
// block j + 1 are multiplied while block j's go through their exponentials (phase A, 48
// matrix instructions with two steps of the softmax behind each), then the values of
// block j with the maxima of block j + 1 and the next loads between (phase B).  48
// queries a wave because LDS is the tightest resource: a key or value read from it is
// multiplied by three times 16 queries.  (64 queries are 256 accumulators, 128 registers of
// queries and 48 of scores, more than there are.)
//
// 8 x 2047 tokens, 10 heads: 185-200 us where all rows are full (0.9 PFLOP/s of the visible
// pairs), 155 left-padded by 0 to half; 290-320 and 290 with 32 queries a wave on
// v_mfma_f32_32x32x16_bf16, tiles of 64 keys through registers, scores, softmax and values
// one after the other, a row to an XCD.  What is left: a block takes 2450 cycles where its
// matrix instructions take 1540 (what is issued between them counts in full from two
// instructions on), and 18000 before the first (the queries' way from memory, all
// workgroups at once, and their rotation).
//
// What a block does around that for a prompt -- rotary embedding, the ring cache
// it leaves -- is attn_prompt_prepare_kernel at
// the end of this file; the queries take their rotary embedding inside the
// attention kernel.
#include "rg_common.h"
#include "rg_internal.h"
#include "rg_matrix_asm.h"

namespace rg {
namespace {

#define RG_INLINE __attribute__((always_inline))
constexpr int kAttnHd = 256;
constexpr int kBlockKeys = 32;
constexpr int kBlockBytes = kBlockKeys * kAttnHd * 2;
constexpr int kRing = 4;  // blocks of keys, and of values, in LDS
constexpr int kAttnLds = 2 * kRing * kBlockBytes;

using namespace matrix_asm;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;

union AFrag {
  bf16x8 v;
  f32x4 q;
  uint32_t u[4];
};

// The output accumulators of a lane (O^T: 16 blocks of 16 dimensions by QB blocks of 16
// queries, 4 registers each) live in the accumulation registers a[0:255] for the whole
// kernel, written and read by inline assembly with the register numbers spelled out:
// nothing but the second product, the rare rescaling and the final store touches them
// (left to the register allocator they were moved between the two register files every
// block).  The build checks that the compiler allocates no accumulation register of its
// own in this file.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// Rotary embedding of the first half of a query's dimensions (elements i and
// i + 64, i < 64) where the query lies as operand fragments: k-steps 0 and 1 hold
// this lane's elements 32 ks + 8 quarter + 0..7, k-steps 2 and 3 their partners.
// `table` is the lane's share of the query's row of sines and cosines (see
// attn_prompt_prepare_kernel).  The arithmetic of rg_rope_pair, element for
// element: products and sums rounded one by one.
__device__ __forceinline__ void rotate_query(AFrag (&qf)[8], const u32x4 (&table)[4]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      float vlo[2], vhi[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t sc = table[2 * ks + (w >> 1)][2 * (w & 1) + e];
        const float sn = __uint_as_float(sc << 16);
        const float cs = __uint_as_float(sc & 0xffff0000u);
        const uint32_t l = qf[ks].u[w], h = qf[ks + 2].u[w];
        const float lo = __uint_as_float(e == 0 ? l << 16 : l & 0xffff0000u);
        const float hi = __uint_as_float(e == 0 ? h << 16 : h & 0xffff0000u);
        vlo[e] = round_to_bf16(lo * cs) - round_to_bf16(hi * sn);
        vhi[e] = round_to_bf16(hi * cs) + round_to_bf16(lo * sn);
      }
      qf[ks].u[w] = pack_bf16x2(vlo[0], vlo[1]);
      qf[ks + 2].u[w] = pack_bf16x2(vhi[0], vhi[1]);
    }
  }
}

// Below every score that is a number, in units of log2: the running maximum before a
// query's first visible key (a masked score is minus infinity).
constexpr float kNoMaximum = -3.0e38f;

// ROPE: the queries come before their rotary embedding and take it here, in
// the registers they are loaded to (p.rope_table); a pass of its own over them
// reads and writes every query once more (8 x 2047 tokens, 10 heads: 43 us).
// COLUMNS: the values come transposed, [row, 256, T_pad], else key by key.  Launched as
// rotated and key by key, or as neither.
// QB: blocks of 16 queries per wave.
template <bool ROPE, bool COLUMNS, int QB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
attn_prefill_bf16_kernel(AttnPrefillArgs p) {
  extern __shared__ __align__(16) unsigned char attn_lds[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte*)attn_lds;
  constexpr int kQ = 16 * QB;       // queries per wave
  constexpr int kMfmas = 16 * QB;   // of either product, per block of keys

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 15, quarter = lane >> 4;
  const int T = p.T, H = p.H;
  const int units = (T + kQ - 1) / kQ * H;  // (query tile, head) pairs of a row
  const int groups = (units + 3) / 4;
  // The longest workgroups (last query tiles) of all rows first.  Workgroups go to the
  // eight XCDs in turn, each with an L2 of its own; which row an XCD gets turns every
  // eight ranks: its 32 workgroups read a few rows' keys and values, and the XCDs'
  // shares come out alike where rows differ (8 x 2047 tokens, left-padded by 0 to 966:
  // 174 -> 155 us; a row to an XCD is 2 % better where all are full).
  const int rank = (int)(blockIdx.x / p.B);
  const int b = (int)((blockIdx.x % p.B + rank / 8) % p.B);
  const int first_unit = 4 * (groups - 1 - rank);
  const int last_unit = first_unit + 3 < units ? first_unit + 3 : units - 1;
  const int unit = first_unit + wave;
  const bool works = unit < units;
  const int q0 = (works ? unit : units - 1) / H * kQ;  // this wave's first query
  const int head = (works ? unit : units - 1) % H;

  // descriptors over this row's tensors
  const uint32_t q_row_bytes = (uint32_t)H * kAttnHd * 2u;
  const __amdgpu_buffer_rsrc_t rq =
      make_rsrc((const char*)p.q + (int64_t)b * T * q_row_bytes,
                (uint32_t)T * q_row_bytes);
  const __amdgpu_buffer_rsrc_t rlo = make_rsrc(
      (const char*)p.lo + (int64_t)b * T * 4, (uint32_t)T * 4u);
  const u32x4 rk = scalar_rsrc((const char*)p.k + (int64_t)b * T * (kAttnHd * 2),
                               (uint32_t)T * (kAttnHd * 2u));
  const uint32_t v_row_bytes = COLUMNS ? (uint32_t)p.T_pad * 2u : kAttnHd * 2u;
  const uint32_t v_bytes = (COLUMNS ? (uint32_t)kAttnHd : (uint32_t)T) * v_row_bytes;
  const u32x4 rv = scalar_rsrc((const char*)p.v + (int64_t)b * v_bytes, v_bytes);

  // ---- everything that is asked for at once: which keys are seen, the queries (the B
  //      operand of the first product, 8 k-steps of 32 dimensions) and their rotation;
  //      queries past the end read as zero ------------------------------------------
  auto lo_at = [&](int t) RG_INLINE {
    return (int)__builtin_amdgcn_raw_buffer_load_b32(
        rlo, t < T ? (uint32_t)t * 4u : kBufferOutOfRange, 0, 0);
  };
  const int q_last = q0 + kQ - 1 < T - 1 ? q0 + kQ - 1 : T - 1;
  const int lo_raw[3] = {lo_at(first_unit / H * kQ), lo_at(q0), lo_at(q_last)};
  __builtin_amdgcn_sched_barrier(0);
  AFrag qf[QB][8];
  u32x4 table[ROPE ? QB : 1][4];
  int lo_q[QB];
  const __amdgpu_buffer_rsrc_t rt =
      make_rsrc((const char*)p.rope_table + (int64_t)b * T * 256, ROPE ? (uint32_t)T * 256u : 0u);
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int q = q0 + 16 * qb + n;
    const uint32_t off = (uint32_t)q * q_row_bytes + (uint32_t)head * 512u + 16u * quarter;
    lo_q[qb] = lo_at(q);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      qf[qb][ks].q = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     rq, q < T ? off + 64u * ks : kBufferOutOfRange, 0, 0));
    if constexpr (ROPE) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        table[qb][i] = __builtin_amdgcn_raw_buffer_load_b128(
            rt,
            q < T ? (uint32_t)q * 256u + 32u * quarter + 128u * (i >> 1) + 16u * (i & 1)
                  : kBufferOutOfRange,
            0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  take_accumulators();
  for_n<64 * QB>([&](auto I) RG_INLINE { acc_zero<decltype(I)::value>(); });

  // first visible key of a query (non-decreasing in it): what bounds the blocks that
  // the workgroup and this wave need
  auto uniform = [](int v) RG_INLINE { return __builtin_amdgcn_readfirstlane(v); };
  const int lo_group = uniform(lo_raw[0]), lo_first = uniform(lo_raw[1]);
  const int lo_last = uniform(lo_raw[2]);
  const int group_last = last_unit / H * kQ + kQ - 1;
  const int j_begin = lo_group / kBlockKeys;
  const int j_end = (group_last < T - 1 ? group_last : T - 1) / kBlockKeys;  // inclusive
  const int j_first = works ? lo_first / kBlockKeys : 0x7fffffff;
  const int j_last = works ? q_last / kBlockKeys : -1;

  // ---- blocks of keys and values into LDS ------------------------------------------
  // A load instruction fills 1 KB.  Keys (and values key by key): two rows, 32 chunks of
  // 16 bytes each, permuted by the row's number; a wave's four instructions take rows
  // 8 r + 2 wave and the next.  Values in columns: 16 rows of a dimension, 64 bytes.
  const int row2 = 2 * wave + (lane >> 5);
  const uint32_t vk = (uint32_t)(row2 * 512 + 16 * ((lane & 31) ^ row2));
  const uint32_t vv =
      COLUMNS ? (uint32_t)(16 * wave + (lane >> 2)) * v_row_bytes +
                    16u * ((lane & 3) ^ ((lane >> 3) & 3))
              : (uint32_t)(row2 * 512 + 16 * ((lane & 31) ^ ((row2 & 3) << 1)));
  auto load_one = [&](int to, int r, uint32_t v, u32x4 rsrc, int at) RG_INLINE {
    const uint32_t where = lds0 + (uint32_t)to + 4096u * (uint32_t)r + 1024u * (uint32_t)wave;
    load_lds_16<0>(where, v, rsrc, at);
  };
  // (past the last key the descriptor's end: nothing is read)
  auto load_keys = [&](int j, int r) RG_INLINE {
    load_one((j & (kRing - 1)) * kBlockBytes, r, vk, rk, (j * kBlockKeys + 8 * r) * 512);
  };
  auto load_values = [&](int j, int r) RG_INLINE {
    const int to = (kRing + (j & (kRing - 1))) * kBlockBytes;
    if (COLUMNS) {
      // (columns behind T_pad belong to the next dimension: not asked for)
      const bool there = j * kBlockKeys < p.T_pad;
      load_one(to, r, there ? vv : kBufferOutOfRange, rv,
               there ? 64 * r * (int)v_row_bytes + j * kBlockKeys * 2 : 0);
    } else {
      load_one(to, r, vv, rv, (j * kBlockKeys + 8 * r) * 512);
    }
  };

#pragma unroll
  for (int i = 0; i < 20; ++i) {
    const int r = i & 3;
    if (i < 8) load_keys(j_begin + i / 4, r);
    else if (i < 12) load_values(j_begin, r);
    else if (i < 16) load_keys(j_begin + 2, r);
    else load_values(j_begin + 1, r);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < 4) load_keys(j_begin + 3, i);
    else load_values(j_begin + 2, i - 4);
  if constexpr (ROPE)
    for_n<QB>([&](auto I) RG_INLINE {
      rotate_query(qf[decltype(I)::value], table[decltype(I)::value]);
    });
  float m_run[QB], l_run[QB];  // running maximum (units of log2), this quarter's sum
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = kNoMaximum;
    l_run[qb] = 0.0f;
  }
  const float scale_log2 = __uint_as_float(
      (uint32_t)uniform((int)__float_as_uint(p.scale * kLog2e)));

  // ---- operands from LDS ---------------------------------------------------------------
  // (kept from being spread over a register per constant offset)
  uint32_t k_lane = lds0 + (uint32_t)(512 * n + 16 * (quarter ^ (n & 7)));
  uint32_t v_lane =
      lds0 + kRing * kBlockBytes +
      (COLUMNS ? (uint32_t)(64 * n + 16 * ((quarter >> 1) ^ ((n >> 1) & 3)) + 8 * (quarter & 1))
               : (uint32_t)(512 * (4 * quarter + (n >> 2)) +
                            16 * (((n & 3) >> 1) ^ ((n >> 2) << 1)) + 8 * (n & 1)));
  constexpr int kAhead = 3;  // fragments on their way
  constexpr int kFrags = kAhead + 1;
  f32x4 ring[kFrags];
  // fragment f of a block of keys: keys 16 (f / 8) .., k-step f % 8 (the second 16 keys'
  // scores are started when half of the block before has left its registers)
  auto read_keys = [&](int j, auto F) RG_INLINE {
    constexpr int f = decltype(F)::value, ks = f % 8;
    const uint32_t at = (k_lane ^ (64u * (ks & 1))) + (uint32_t)((j & (kRing - 1)) * kBlockBytes);
    ring[f % kFrags] = *reinterpret_cast<const lds_f32x4*>(
        (lds_byte*)(uintptr_t)at + 128 * (ks >> 1) + 8192 * (f / 8));
  };
  // fragment d of a block of values: dimensions 16 d ..
  auto read_values = [&](int j, auto D) RG_INLINE {
    constexpr int d = decltype(D)::value;
    const uint32_t to = (uint32_t)((j & (kRing - 1)) * kBlockBytes);
    if constexpr (COLUMNS) {
      union {
        u32x2 h[2];
        f32x4 v;
      } u;
      const uint32_t at = v_lane + to;
      u.h[0] = *reinterpret_cast<const lds_u32x2*>((lds_byte*)(uintptr_t)at + 1024 * d);
      u.h[1] = *reinterpret_cast<const lds_u32x2*>((lds_byte*)(uintptr_t)(at ^ 32u) + 1024 * d);
      ring[d % kFrags] = u.v;
    } else {
      union {
        s16x4 h[2];
        f32x4 v;
      } u;
      lds_byte* const at =
          (lds_byte*)(uintptr_t)((v_lane ^ (32u * (d & 3))) + to) + 128 * (d >> 2);
      u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
      u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 8192));
      ring[d % kFrags] = u.v;
    }
  };

  // ---- one block of keys -------------------------------------------------------------
  // s[kb][qb]: S^T of 16 keys by 16 queries
  using Scores = f32x4[2][QB];
  auto score_mfma = [&](Scores& s, auto I) RG_INLINE {
    constexpr int i = decltype(I)::value, f = i / QB, qb = i % QB, ks = f % 8;
    f32x4& c = s[f / 8][qb];
    const f32x4 &k = ring[f % kFrags], &q = qf[qb][ks].q;
    if constexpr (ks == 0)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(k), "v"(q));
    else
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(k), "v"(q));
  };
  AFrag pf[QB];
  // Scores 2 i and 2 i + 1 of a query block, i = 0..3, to probabilities, in seven steps:
  // a matrix instruction leaves room for two others before the next, and a longer run
  // of them leaves the matrix pipe idle (all seven behind every fourth: a block's loop
  // 2630 cycles).
  constexpr int kSteps = 7 * 4 * QB;
  float p0, p1;
  auto probability_step = [&](const Scores& s, auto I) RG_INLINE {
    constexpr int o = decltype(I)::value / 7, step = decltype(I)::value % 7;
    constexpr int qb = o / 2 % QB, i = o % 2 + 2 * (o / (2 * QB));  // 16 keys after 16
    if constexpr (step < 2) {
      float& x = step ? p1 : p0;
      x = __builtin_fmaf(s[i >> 1][qb][2 * (i & 1) + step], scale_log2, -m_run[qb]);
    }
    if constexpr (step == 2) p0 = __builtin_amdgcn_exp2f(p0);
    if constexpr (step == 3) p1 = __builtin_amdgcn_exp2f(p1);
    if constexpr (step == 4) l_run[qb] += p0;
    if constexpr (step == 5) l_run[qb] += p1;
    if constexpr (step == 6) pf[qb].u[i] = pack_bf16x2(p0, p1);
  };
  auto value_mfma = [&](auto I) RG_INLINE {
    constexpr int i = decltype(I)::value;
    acc_mfma<i>(ring[i / QB % kFrags], pf[i % QB].q);
  };
  auto mask = [&](Scores& s, int j) RG_INLINE {  // where the band's edges cross the block
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int n = ln & 15, quarter = ln >> 4;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int q = q0 + 16 * qb + n, lo = lo_q[qb];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = j * kBlockKeys + 16 * kb + 4 * quarter + r;
          s[kb][qb][r] = key >= lo && key <= q ? s[kb][qb][r] : -__builtin_inff();
        }
    }
  };
  auto interior = [&](int j) RG_INLINE {
    return j * kBlockKeys + kBlockKeys - 1 <= q0 && j * kBlockKeys >= lo_last;
  };
  // The running maximum moves only when a block's exceeds it by more than 2^8: the
  // accumulators are rescaled rarely.
  float most[QB];  // the next block's maxima, of this lane's scores
  auto maximum = [&](const Scores& s, auto QBI) RG_INLINE {
    constexpr int qb = decltype(QBI)::value;
    const f32x4 &a = s[0][qb], &c = s[1][qb];
    most[qb] = max3(max3(a[0], a[1], a[2]), max3(a[3], c[0], c[1]), fmaxf(c[2], c[3]));
  };
  auto rescale_where_needed = [&](bool first_block) RG_INLINE {
    float over = __builtin_fmaf(most[0], scale_log2, -m_run[0]);
#pragma unroll
    for (int qb = 1; qb < QB; ++qb)
      over = fmaxf(over, __builtin_fmaf(most[qb], scale_log2, -m_run[qb]));
    if (__builtin_expect(__ballot(over > 8.0f) == 0, 1)) return;
    float alpha[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float m = most[qb] * scale_log2;  // (the scale is positive)
      m = fmaxf(m, __shfl_xor(m, 16));
      m = fmaxf(m, __shfl_xor(m, 32));
      m = fmaxf(m, m_run[qb]);
      alpha[qb] = __builtin_amdgcn_exp2f(m_run[qb] - m);
      m_run[qb] = m;
      l_run[qb] *= alpha[qb];
    }
    if (first_block) return;  // (the accumulators are zeros)
    wait_for_matrix_results();
    for_n<64 * QB>([&](auto I) RG_INLINE {
      constexpr int i = decltype(I)::value;
      acc_write<i>(acc_read<i>() * alpha[i / 4 % QB]);
    });
  };
  auto settle = [&](Scores& s) RG_INLINE {  // results of the matrix instructions before this
    wait_for_matrix_results();
#pragma unroll
    for (int i = 0; i < 2 * QB; ++i) asm volatile("" : "+v"(s[i / QB][i % QB]));
  };
  auto scores_alone = [&](Scores& s, int j) RG_INLINE {
    for_n<kAhead>([&](auto F) RG_INLINE { read_keys(j, F); });
    for_n<16>([&](auto F) RG_INLINE {
      constexpr int f = decltype(F)::value;
      if constexpr (f + kAhead < 16) read_keys(j, std::integral_constant<int, f + kAhead>{});
      for_n<QB>([&](auto K) RG_INLINE {
        score_mfma(s, std::integral_constant<int, f * QB + decltype(K)::value>{});
      });
    });
    settle(s);
    if (!interior(j)) mask(s, j);
    for_n<QB>([&](auto I) RG_INLINE { maximum(s, I); });
  };
  // Behind this every wave is done with the keys of block j + 1 and the values of
  // j - 1, and keys j + 2 and values j + 1 are in LDS (the loads of one round may be on
  // their way).
  auto block_barrier = [&] RG_INLINE { asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory"); };
  auto load = [&](int j, int i) RG_INLINE {  // the i-th of a round's eight
    if (i < 4) load_keys(j + 4, i);
    else load_values(j + 3, i - 4);
  };
  // Probabilities and values of block j, scores of block j + 1.
  auto block = [&](int j, Scores& now, Scores& next) RG_INLINE {
    const bool values = j >= j_first && j <= j_last;
    const bool scores = j + 1 >= j_first && j + 1 <= j_last;
    asm volatile("" : "+v"(k_lane), "+v"(v_lane));
    if (__builtin_expect(values && scores, 1)) {
      for_n<kMfmas>([&](auto I) RG_INLINE {
        constexpr int i = decltype(I)::value, f = i / QB;
        score_mfma(next, I);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i % QB == 0) {
          if constexpr (f + kAhead < 16) read_keys(j + 1, std::integral_constant<int, f + kAhead>{});
          else read_values(j, std::integral_constant<int, f + kAhead - 16>{});
        }
        constexpr int from = i * kSteps / kMfmas, to = (i + 1) * kSteps / kMfmas;
        for_n<to - from>([&](auto S) RG_INLINE {
          probability_step(now, std::integral_constant<int, from + decltype(S)::value>{});
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      const bool edge = !interior(j + 1);
      for_n<kMfmas>([&](auto I) RG_INLINE {
        constexpr int i = decltype(I)::value, d = i / QB;
        value_mfma(I);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i == 8 * QB) block_barrier();
        if constexpr (i % QB == 0) {
          if constexpr (d + kAhead < 16) read_values(j, std::integral_constant<int, d + kAhead>{});
          else read_keys(j + 2, std::integral_constant<int, d + kAhead - 16>{});
        }
        if constexpr (i == 6 * QB) {
#pragma unroll
          for (int k = 0; k < 2 * QB; ++k) asm volatile("" : "+v"(next[k / QB][k % QB]));
          if (__builtin_expect(edge, 0)) mask(next, j + 1);
        }
        if constexpr (i > 6 * QB && i % 2 == 1 && (i - 6 * QB) / 2 < QB)
          maximum(next, std::integral_constant<int, (i - 6 * QB) / 2>{});
        if constexpr (i > 8 * QB && i <= 8 * QB + 16 && i % 2 == 1)
          load(j, (i - 8 * QB) / 2);
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      if (values) {
        for_n<kSteps>([&](auto I) RG_INLINE { probability_step(now, I); });
        for_n<kAhead>([&](auto D) RG_INLINE { read_values(j, D); });
        for_n<16>([&](auto D) RG_INLINE {
          constexpr int d = decltype(D)::value;
          if constexpr (d + kAhead < 16) read_values(j, std::integral_constant<int, d + kAhead>{});
          for_n<QB>([&](auto K) RG_INLINE {
            value_mfma(std::integral_constant<int, d * QB + decltype(K)::value>{});
          });
        });
      }
      if (scores) scores_alone(next, j + 1);
      block_barrier();
      for (int i = 0; i < 8; ++i) load(j, i);
      for_n<kAhead>([&](auto F) RG_INLINE { read_keys(j + 2, F); });
    }
    if (scores) rescale_where_needed(j + 1 == j_first);
  };

  Scores even, odd;
#pragma unroll
  for (int i = 0; i < 2 * QB; ++i)
    even[i / QB][i % QB] = odd[i / QB][i % QB] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  if (j_first == j_begin) {
    scores_alone(even, j_begin);
    rescale_where_needed(true);
  }
  for_n<kAhead>([&](auto F) RG_INLINE { read_keys(j_begin + 1, F); });
  for (int j = j_begin; j <= j_end; j += 2) {
    block(j, even, odd);
    if (j + 1 > j_end) break;
    block(j + 1, odd, even);
  }
  // (no load outlives the workgroup's LDS)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (!works) return;

  // ---- normalise and store: a lane's query of each block, dimensions 16 d + 4 quarter
  //      .. + 3; two neighbouring quarters trade runs of two blocks for eight in a row --
  wait_for_matrix_results();
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(
      (char*)p.out + (int64_t)b * T * q_row_bytes, (uint32_t)T * q_row_bytes);
  for_n<QB>([&](auto QBI) RG_INLINE {
    constexpr int qb = decltype(QBI)::value;
    float l = l_run[qb];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const int q = q0 + 16 * qb + (ln & 15);
    const uint32_t off = (uint32_t)q * q_row_bytes + (uint32_t)head * 512u +
                         2u * (uint32_t)(ln & 16) + 8u * (uint32_t)(ln >> 4 & 2);
    for_n<8>([&](auto P) RG_INLINE {
      constexpr int pair = decltype(P)::value;
      uint32_t w[2][2];
      for_n<4>([&](auto E) RG_INLINE {
        constexpr int e = decltype(E)::value, at = 4 * ((2 * pair + e / 2) * QB + qb) + 2 * (e % 2);
        w[e / 2][e % 2] = pack_bf16x2(acc_read<at>() * inv, acc_read<at + 1>() * inv);
      });
      const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
      buffer_store_16(u32x4{s0[0], s1[0], s0[1], s1[1]}, ro,
                      q < T ? off + 64u * pair : kBufferOutOfRange, 0);
    });
  });
}

// ---------------------------------------------------------------- prepare --
// Everything of the block between its projections and the attention kernel,
// in one pass over the keys (recurrentgemma/torch/modules.py:431-440
// and the ring cache of a prompt, :253-283): rotary embedding of the keys, the
// sines and cosines the queries are rotated with (one word per token and pair:
// sine in the low half, cosine in the high half, bf16), the last min(window, T)
// keys and values in their ring slots, zeros in the slots never written, and
// the token count.
//
// One workgroup per (row, 32 tokens and 32 ring slots), which leaves the chip
// full from 8 x 1024 tokens on.  Bound by memory (8 x 2047 tokens: 17 MB in,
// 30 MB out); the tensor operations it replaces were ten launches, 146 us
// there.
constexpr int kPrepTokens = 32;

__device__ __forceinline__ int64_t position_at(const AttnPromptArgs& p,
                                               int64_t i) {
  return p.pos_kind == kSegI64
             ? reinterpret_cast<const int64_t*>(p.pos)[i]
             : (int64_t)reinterpret_cast<const int32_t*>(p.pos)[i];
}

__global__ void __launch_bounds__(256)
attn_prompt_prepare_kernel(AttnPromptArgs p) {
#pragma clang fp contract(off)
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
  // values, to their ring slots
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int t = t0 + 8 * j + tid / 32;
    const int slot = t < T ? slot_of(t) : -1;
    if (slot >= 0) {
      const int d = 8 * (tid % 32);
      *reinterpret_cast<u32x4*>(ring_v + (int64_t)slot * kAttnHd + d) =
          *reinterpret_cast<const u32x4*>(v + (int64_t)t * kAttnHd + d);
    }
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
  const int64_t tokens = a.ring_k && a.window > a.T ? a.window : a.T;
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

namespace {
template <bool ROPE, bool COLUMNS, int QB>
hipError_t launch_prefill(const AttnPrefillArgs& a, hipStream_t s) {
  const int64_t units = (int64_t)((a.T + 16 * QB - 1) / (16 * QB)) * a.H;
  const int64_t blocks = (units + 3) / 4 * a.B;
  if (blocks <= 0 || blocks > 0x7fffffff || units > 0x7ffffff0) return hipErrorInvalidValue;
  static OncePerDevice once;
  const auto kernel = attn_prefill_bf16_kernel<ROPE, COLUMNS, QB>;
  hipError_t e = set_max_dynamic_lds(once, (const void*)kernel, kAttnLds);
  if (e != hipSuccess) return e;
  kernel<<<dim3((unsigned)blocks), 256, kAttnLds, s>>>(a);
  return hipGetLastError();
}
}  // namespace

namespace {
template <int QB>
hipError_t launch_queries(const AttnPrefillArgs& a, hipStream_t s) {
  if (a.T_pad > 0) return launch_prefill<false, true, QB>(a, s);
  if (!a.rope_table) return hipErrorInvalidValue;
  return launch_prefill<true, false, QB>(a, s);
}
// 32 queries a wave up to two rounds of the chip of them: half as many workgroups again,
// each with two thirds of the work (us with 48 / 32, 10 heads: 1 x 300 tokens 28 / 22,
// 1 x 2047 86 / 67, 4 x 1000 58 / 47, 8 x 700 50 / 47; 16 heads 1 x 1000 52 / 41, 4 x 1000
// 60 / 59, 3 x 1500 78 / 79).
bool short_tiles(const AttnPrefillArgs& a) {
  const int64_t units = (int64_t)((a.T + 31) / 32) * a.H;
  return (units + 3) / 4 * a.B <= 512;
}
}  // namespace

hipError_t launch_attn_prefill_bf16(const AttnPrefillArgs& a, hipStream_t s) {
  // needs head dimension 256 and rows whose byte offsets fit 32 bits (checked by the
  // caller); values in columns T_pad (a multiple of 64) long, or key by key (T_pad 0):
  // then the queries take their rotary embedding here
  return short_tiles(a) ? launch_queries<2>(a, s) : launch_queries<3>(a, s);
}

}  // namespace rg
