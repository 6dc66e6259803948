// Whole recurrent core of a prefill in one launch (bf16, 256-wide heads), the
// form with TWO waves per SIMD that take turns at the matrix unit and at the
// vector unit.
//
// One workgroup of eight waves per (sequence row b, head h).  Wave w owns 32
// channels of the head for both gates; its 2 x 256 x 32 weights (128
// accumulation registers) stay resident.  The waves form two teams (0-3 and
// 4-7, one wave of each per SIMD) that walk the sequence in blocks of 32
// tokens, each block in two phases:
//   M  the 32 matrix instructions of the block (pre-activations of both
//      gates), with little else to issue: this wave's share of the conv of
//      the next block, the stores of the block before, the next loads, and
//      at the end a part of the gate arithmetic;
//   G  the rest of the gate arithmetic and the recurrence of the block:
//      vector instructions only.
// Team 1 runs one phase behind team 0, a workgroup barrier after every phase
// keeps it there: while one wave of a SIMD is in G the other is in M, so the
// matrix instructions and their operand reads issue in the gaps of the other
// wave's arithmetic instead of in its own instruction stream.  (With both
// waves of a SIMD in the same phase the kernel is a fifth slower; with the
// wave in M not raised in priority over the one in G, a tenth.)  Same
// arithmetic in the same order as the one-wave-per-SIMD form in rg_prefill.hip:
// the two give bit-identical results.
//
// Whole rows and rows in chunks, with or without the block's GELU join; needs
// the weights re-laid-out (rg_pack_gate_weights): the launcher in
// rg_prefill.hip sends callers without them to the other form.
//
// Replaces the chain Conv1D.forward -> RGLRU.forward of
// recurrentgemma/torch/modules.py:632-643 (layers.py:447-529, 313-365,
// 140-191) for prefill.
#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"
#include "rg_two_teams.h"

namespace rg {
namespace {

using namespace two_teams;

constexpr int kTM = 64;    // tokens per raw tile (two blocks)
// Raw x of a 64-token tile as the memory pipe writes it into LDS: rows -4 ..
// 63 of the tile, 512 bytes each; two tiles.
constexpr int kRawRows = kTM + kRawHalo;
constexpr int kRawLoads = kRawRows / 2;
constexpr int kRawLoadsPerWave = (kRawLoads + kWaves - 1) / kWaves;
constexpr int kRawTileBytes = kRawLoadsPerWave * kWaves * 2 * kRawRowBytes;
constexpr int kXcOff = 0;
constexpr int kRawOff = kXcOff + kXcRing * kXcBlockBytes;
constexpr int kPatchOff = kRawOff + 2 * kRawTileBytes;
constexpr int kConvTabOff = kPatchOff + kWaves * kPatchBytesPerWave;
constexpr int kTeamsLdsBytes = kConvTabOff + kConvTabBytes;
static_assert(kTeamsLdsBytes <= 160 * 1024, "LDS of one CU");

// What one workgroup does with its tiles.  A row cut into chunks takes two
// launches: the first runs chunk 0 as kChunkHead and chunks 1 .. n-2 as
// kChunkSummary side by side, the second chunks 1 .. n-1 as kChunkReplay,
// each starting from the summaries of the chunks before it.
enum PrefillMode {
  kWholeRow = 0,      // a whole row of one head: y, h_last, conv state
  kChunkSummary = 1,  // a chunk from a zero state: (prod a, h_end), no y
  kChunkReplay = 2,   // a chunk from its incoming state: y, ...
  kChunkHead = 3      // chunk 0 from h0: y, and its end state as a summary
};

// GELU: y is written as y * gelu(gate_branch), the join of the recurrent
// block's two branches (recurrentgemma/torch/modules.py:627-628, 644),
// instead of the plain RG-LRU output.
template <int MODE, bool GELU>
__device__ __forceinline__ void prefill_teams_body(const FusedArgs& p,
                                                   const int chunk) {
  // how much of the gate arithmetic runs at the end of phase M (with the
  // join, phase G carries 13 more vector slots per element)
  constexpr int kTailX = GELU ? kTailXJoined : kTailXPlain;
  constexpr int kTailA = GELU ? kTailAJoined : kTailAPlain;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  lds_byte* const lds3 = (lds_byte*)lds_raw;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int team = wave >> 2;
  const int in_team = wave & 3;
  const int b = blockIdx.x / p.H;
  const int h = blockIdx.x % p.H;
  const int T_len = p.T;
  const int64_t W = p.W;
  const int ntiles = (T_len + kTM - 1) / kTM;  // of the whole row
  const int tile_begin = MODE == kWholeRow ? 0 : chunk * p.tiles_per_chunk;
  int tile_end = MODE == kWholeRow ? ntiles : tile_begin + p.tiles_per_chunk;
  if (tile_end > ntiles) tile_end = ntiles;
  const bool last_chunk = tile_end == ntiles;
  const bool upper = lane >= 32;
  const int n0 = wave * 32;  // first channel of this wave in the head

  // ---- addressing -----------------------------------------------------------
  const uint32_t row_bytes = 2u * (uint32_t)p.W;
  const uint32_t seq_bytes = (uint32_t)T_len * row_bytes;  // < 2^31 (launcher)
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc((const char*)p.x + (int64_t)b * seq_bytes, seq_bytes);
  const __amdgpu_buffer_rsrc_t ry = make_rsrc(
      (char*)p.y + (int64_t)b * seq_bytes, MODE == kChunkSummary ? 0 : seq_bytes);
  // GELU: the block's other branch, read where y is written
  const __amdgpu_buffer_rsrc_t rgate = make_rsrc(
      (const char*)p.gate_branch + (int64_t)b * seq_bytes,
      GELU && MODE != kChunkSummary ? seq_bytes : 0);
  const bool seg_is64 = p.seg_kind == kSegI64;
  const uint32_t seg_esize = seg_is64 ? 8u : 4u;
  const __amdgpu_buffer_rsrc_t rseg =
      make_rsrc((const char*)p.segpos + (int64_t)b * T_len * seg_esize,
                (uint32_t)T_len * seg_esize);

  // Document starts of a tile: lane j looks at token 64*tile + j.
  uint32_t seg_lo = 1, seg_hi = 0;
  auto fetch_seg = [&](int tile) {
    const int t = tile * kTM + lane;
    const uint32_t off = (tile >= 0 && tile < ntiles && t < T_len)
                             ? (uint32_t)t * seg_esize
                             : kBufferOutOfRange;
    seg_lo = __builtin_amdgcn_raw_buffer_load_b32(rseg, off, 0, 0);
    seg_hi = __builtin_amdgcn_raw_buffer_load_b32(
        rseg, seg_is64 ? off + 4u : kBufferOutOfRange, 0, 0);
  };
  auto start_mask = [&](int tile) -> uint64_t {
    uint32_t lo = seg_lo, hi = seg_hi;
    asm volatile("" : "+v"(lo), "+v"(hi));
    const int t = tile * kTM + lane;
    return __ballot(tile >= 0 && tile < ntiles && t < T_len && (lo | hi) == 0u);
  };

  // Raw x of one tile -> LDS by the memory pipe: 34 wave-wide loads of two
  // rows each, five per wave (the six beyond 34 are sent out of range and
  // fill padding rows with zeros).
  const uint32_t dma_lane_off =
      2u * (uint32_t)(h * kBW) + 16u * (uint32_t)(lane & 31);
  auto dma_tile = [&](int tile, int j) {  // this wave's load j of the tile
    lds_byte* const dst = lds3 + kRawOff + (tile & 1) * kRawTileBytes;
    const int t0 = tile * kTM - kRawHalo + (lane >> 5);
    const int i = wave + kWaves * j;
    uint32_t voff = (uint32_t)((t0 + 2 * i) * (int)row_bytes) + dma_lane_off;
    if (kWaves * j + kWaves > kRawLoads)
      voff = i < kRawLoads ? voff : kBufferOutOfRange;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, dst + i * 1024, 16, voff, 0, 0,
                                             0);
  };

  // ---- lane-dependent LDS offsets -------------------------------------------
  // conv: thread -> (channel pair tid % 128, rows 8 rg4 .. 8 rg4 + 7 of a
  // block); team 0 holds row groups 0 and 1, team 1 groups 2 and 3.  Row r of
  // a tile lies at raw row r + kRawHalo; the lane offset points three rows
  // before the group's first.
  const int rg4 = team * 2 + (in_team >> 1);  // 0..3
  const int conv_pair_of_lane = (in_team & 1) * 64 + lane;
  const uint32_t conv_raw_lane =
      kRawOff + (uint32_t)(rg4 * kConvRows + kRawHalo - 3) * kRawRowBytes +
      conv_pair_of_lane * 4;
  // Conv output of token t of a block lies in row xc_row(t): the rows are the
  // A operand's, of whose results a lane gets rows 8 j + 4 (lane / 32) + 0..3,
  // j = 0..3.  In this order those are tokens 0..15 for lanes 0-31 and tokens
  // 16..31 for lanes 32-63, a walk of the recurrence in one piece (B16 T8192
  // W4096: 4 us of 765 against four pieces with the halves in turn).  Summaries
  // keep the tokens in their order: rg_prefill.hip multiplies its product of a
  // in the order that gives.
  constexpr bool halves = MODE != kChunkSummary;
  const uint32_t conv_xc_lane =
      kXcOff +
      (uint32_t)(halves ? 16 * (rg4 & 1) + 4 * (rg4 >> 1) : rg4 * kConvRows) *
          kXcRowBytes +
      conv_pair_of_lane * 4;
  // row of a thread's i-th conv row, relative to its first; likewise the token
  // of a lane's i-th result, relative to its first
  auto xc_row = [](int i) { return halves ? 8 * (i >> 2) + (i & 3) : i; };
  auto token = [](int i) { return halves ? i : 8 * (i >> 2) + (i & 3); };
  // gates: lane -> channel n0 + lane % 32, tokens 16 (lane / 32) + ...
  const uint32_t xc_lane = kXcOff + 4u * (lane >> 5) * kXcRowBytes +
                           2u * (uint32_t)(n0 + (lane & 31));
  // MFMA A operand: lane -> token lane % 32, k offset 8 (lane / 32)
  const uint32_t a_lane =
      kXcOff + (uint32_t)(lane & 31) * kXcRowBytes + 16u * (lane >> 5);
  // output patch of this wave: eight tokens of the lower and eight of the upper
  // lanes at a time, written as row 8 (lane / 32) + ..., channel lane % 32; read
  // back as 16-byte row chunks, lane l taking chunk l % 4 of row l / 4
  const uint32_t patch_w_lane = kPatchOff + wave * kPatchBytesPerWave +
                                (uint32_t)(lane >> 5) * kPatchUpper +
                                2u * (lane & 31);
  const uint32_t patch_r_lane = kPatchOff + wave * kPatchBytesPerWave +
                                (uint32_t)(lane >> 5) * kPatchUpper +
                                (uint32_t)((lane >> 2) & 7) * kPatchStride +
                                16u * (lane & 3);
  const uint32_t y_lane_bytes =
      (uint32_t)(16 * (lane >> 5) + ((lane >> 2) & 7)) * row_bytes +
      2u * (uint32_t)(h * kBW + n0) + 16u * (lane & 3);

  // ---- width-4 conv ---------------------------------------------------------
  Conv conv;
  auto load_rows = [&](int kb, ConvRows& cr) {  // of block kb
    conv_load(lds3,
              conv_raw_lane + (uint32_t)((kb >> 1) & 1) * kRawTileBytes +
                  (uint32_t)(kb & 1) * (32 * kRawRowBytes),
              conv_xc_lane + (uint32_t)(kb % kXcRing) * kXcBlockBytes, cr);
  };
  // Document starts among this thread group's rows (3 before + its own) of
  // block kb: m_tile is the start mask of the block's tile, m_before that of
  // the tile before it.
  auto conv_cuts = [&](int kb, uint64_t m_tile, uint64_t m_before) -> uint32_t {
    const uint64_t lo = ((m_tile << 3) | (m_before >> 61)) >> (rg4 * kConvRows);
    const uint64_t hi = m_tile >> (29 + rg4 * kConvRows);
    const uint64_t bits = (kb & 1) ? hi : lo;
    return (uint32_t)bits & ((1u << (kConvRows + 3)) - 1u);
  };

  // ---- state ------------------------------------------------------------------
  const int ch = h * kBW + n0 + (lane & 31);  // this lane's channel
  const float bias_x = -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[0])[ch]);
  const float bias_a = -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[1])[ch]);
  const float inv_decay = inverse_decay(
      (-8.0f * kLog2e) *
      softplus_precise(bf16_bits_to_f32(((const uint16_t*)p.a_param)[ch])));
  float hc = 0.0f;    // carried state of this lane's channel
  float prod = 1.0f;  // kChunkSummary: product of a over this lane's tokens
  if (MODE == kChunkReplay) {
    // state at the start of this chunk from the summaries of the chunks
    // before it: h <- P[k] h + H[k] (the scan operator of
    // recurrentgemma/jax/scan.py:161-187 over chunks); chunk 0 has P = 0 and
    // H = its end state
    const float* sp = p.ws_p + (int64_t)b * p.chunks * W + ch;
    const float* sh = p.ws_h + (int64_t)b * p.chunks * W + ch;
    for (int k = 0; k < chunk; ++k)
      hc = __builtin_fmaf(sp[(int64_t)k * W], hc, sh[(int64_t)k * W]);
  } else if ((MODE == kWholeRow || MODE == kChunkHead) && p.h0) {
    hc = p.h0[(int64_t)b * W + ch];
  }
  f32x16 acc_x, acc_a;
  // conv outputs of the block in phase G, this lane's tokens, as floats
  uint32_t xr[16];
  u32x4 y_pending[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  uint32_t y_pending_row = kBufferOutOfRange;
  // start masks of the tile before the current G block's, of its own, and of
  // the next
  uint64_t m_prev, m_cur, m_next;

  // gate arithmetic on accumulator elements [i0, i1), in place: the input
  // gate's sigmoid; a = exp2(sigmoid(recurrence gate) * decay)
  auto gate_x = [&](int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i)
      acc_x[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(acc_x[i], -kLog2e, bias_x));
#pragma unroll
    for (int i = i0; i < i1; ++i)
      acc_x[i] = __builtin_amdgcn_rcpf(1.0f + acc_x[i]);
  };
  auto gate_a = [&](int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i)
      acc_a[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(acc_a[i], -kLog2e, bias_a));
#pragma unroll
    for (int i = i0; i < i1; ++i)
      acc_a[i] = gate_exponent(acc_a[i], inv_decay);
#pragma unroll
    for (int i = i0; i < i1; ++i)
      acc_a[i] = __builtin_amdgcn_exp2f(acc_a[i]);
  };
  // ---- phase M of block kb ----------------------------------------------------
  auto phase_m = [&](int kb, auto ODD) {
    constexpr bool odd = decltype(ODD)::value;  // kb % 2, at compile time
    // team 1 reads raw rows that it asked for itself two phases ago (team 0
    // waits for its own at the top of phase G)
    if (!odd && team == 1) wait_vmcnt<0>();
    const uint32_t a_at = a_lane + (uint32_t)(kb % kXcRing) * kXcBlockBytes;
    auto a_read = [&](int ks) {
      return *reinterpret_cast<lds_f32x4*>(lds3 + a_at + ks * 32);
    };
    f32x4 a[kARing];
#pragma unroll
    for (int k = 0; k < kARing - 1; ++k) a[k] = a_read(k);
    // the tokens of the block before leave now
    buffer_store_16(y_pending[0], ry, y_lane_bytes, y_pending_row);
    buffer_store_16(y_pending[1], ry, y_lane_bytes,
                    y_pending_row + 8u * row_bytes);
    const uint32_t cuts = odd ? conv_cuts(kb + 1, m_next, m_cur)
                              : conv_cuts(kb + 1, m_cur, m_prev);
    ConvRows cr;
    // the block's conv outputs for the gate arithmetic, this lane's sixteen
    // tokens: each into the high half of a zeroed register -- the bf16 value
    // as a float without a shift
    const uint32_t x_at = xc_lane + (uint32_t)(kb % kXcRing) * kXcBlockBytes;
#define RG_XR(i)                                                            \
  asm volatile("v_mov_b32 %0, 0\n\tds_read_u16_d16_hi %0, %1 offset:%2"      \
               : "=&v"(xr[i])                                                \
               : "v"(x_at), "n"((8 * ((i) >> 2) + ((i) & 3)) * kXcRowBytes));
    __builtin_amdgcn_s_setprio(kMatrixPriority);
    // The 32 matrix instructions of the block, with this wave's conv rows of
    // the next block and (every second block) the loads of the tile after the
    // next between them.
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
      if (ks + kARing - 1 < 16)
        a[(ks + kARing - 1) % kARing] = a_read(ks + kARing - 1);
      mfma_weight_frag(2 * ks, ks == 0, a[ks % kARing], acc_x);
      mfma_weight_frag(2 * ks + 1, ks == 0, a[ks % kARing], acc_a);
      if (ks == 0) load_rows(kb + 1, cr);
      if (ks >= 3 && ks % 3 == 0 && ks / 3 - 1 < kConvRows / 2)
        conv_pair(lds3, conv, cr, ks / 3 - 1, xc_row);
      // (late in the loop, when the conv rows have left their registers)
      if (ks == 13) { RG_XR(0) RG_XR(1) RG_XR(2) RG_XR(3) RG_XR(4) }
      if (ks == 14) { RG_XR(5) RG_XR(6) RG_XR(7) RG_XR(8) RG_XR(9) RG_XR(10) }
      if (ks == 15) { RG_XR(11) RG_XR(12) RG_XR(13) RG_XR(14) RG_XR(15) }
      if (odd) {
        if (ks == 4) dma_tile((kb >> 1) + 2, 0);
        if (ks == 7) dma_tile((kb >> 1) + 2, 1);
        if (ks == 10) dma_tile((kb >> 1) + 2, 2);
        if (ks == 13) dma_tile((kb >> 1) + 2, 3);
        if (ks == 14) dma_tile((kb >> 1) + 2, 4);
        if (ks == 15) fetch_seg((kb >> 1) + 2);
      }
    }
#undef RG_XR
    __builtin_amdgcn_s_setprio(0);
    if (__builtin_expect(cuts != 0, 0)) conv_with_cuts(lds3, conv, cr, cuts, xc_row);
    // the last matrix results land (19 issue slots); every reader of the
    // accumulators is ordered behind this statement
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc_x), "+v"(acc_a));
    // part of the gate arithmetic here, the rest in phase G: split so that
    // the two phases take about as long
    gate_x(0, kTailX);
    gate_a(0, kTailA);
    // (computed here, before the barrier: nothing else orders them)
    asm volatile("" : "+v"(acc_x), "+v"(acc_a));
  };

  // ---- phase G of block kb ----------------------------------------------------
  // The matrix result gives a lane one channel (lane % 32) and 16 tokens, in a
  // row (lanes 0-31 the first half of the block, lanes 32-63 the second) or, for
  // summaries, in runs of four that alternate between the halves.  The recurrence
  // is walked twice: from the carried state (right for lanes 0-31, whose end value
  // goes to lanes 32-63 with one permlane32_swap), then again from each half's own
  // incoming state.
  auto phase_g_as = [&](int kb, auto GENERAL) {
    constexpr bool general = decltype(GENERAL)::value;
    const int t_blk = kb * kBT;
    u32x4 g_pending[2];
    if (GELU) {
      // the gate-branch values at the positions of this block's outputs:
      // asked for now, used at the end of the phase
      g_pending[0] = __builtin_amdgcn_raw_buffer_load_b128(
          rgate, y_lane_bytes + (uint32_t)t_blk * row_bytes, 0, 0);
      g_pending[1] = __builtin_amdgcn_raw_buffer_load_b128(
          rgate, y_lane_bytes + (uint32_t)(t_blk + 8) * row_bytes, 0, 0);
    }
    gate_x(kTailX, 16);
    gate_a(kTailA, 16);
    float xn[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) xn[i] = __uint_as_float(xr[i]) * acc_x[i];
    if (general) {
      // document start: a = 0; past the end of the sequence: a = 1, no input.
      // The input scale sqrt(1 - a^2) comes out as 1 at a start.
      const int first = upper ? (halves ? 16 : 4) : 0;
      const uint32_t starts = (uint32_t)(m_cur >> ((kb & 1) * 32 + first));
      const int left = T_len - t_blk - first;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        acc_a[i] = ((starts >> token(i)) & 1u) ? 0.0f : acc_a[i];
        acc_a[i] = token(i) < left ? acc_a[i] : 1.0f;
        xn[i] = token(i) < left ? xn[i] : 0.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      xn[i] = xn[i] *
              __builtin_amdgcn_sqrtf(__builtin_fmaf(-acc_a[i], acc_a[i], 1.0f));
    // the state from the carried one over elements [i0, i1) of both halves, each
    // handed to keep(i, state); the end state becomes the carried one
    auto walk = [&](int i0, int i1, auto&& keep) {
      float e1 = hc;
#pragma unroll
      for (int i = i0; i < i1; ++i) e1 = __builtin_fmaf(acc_a[i], e1, xn[i]);
      const auto sw = __builtin_amdgcn_permlane32_swap(
          __float_as_uint(hc), __float_as_uint(e1), false, false);
      // lanes 0-31: carry, 32-63: e1 of 0-31
      float hh = __uint_as_float(sw[0]);
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        hh = __builtin_fmaf(acc_a[i], hh, xn[i]);
        keep(i, hh);
      }
      const auto end = __builtin_amdgcn_permlane32_swap(
          __float_as_uint(hh), __float_as_uint(hh), false, false);
      hc = __uint_as_float(end[1]);  // all lanes: end value of 32-63
    };
    if (MODE == kChunkSummary) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        walk(4 * g, 4 * g + 4, [&](int i, float) { prod *= acc_a[i]; });
    } else {
      float hv[4];
      walk(0, 16, [&](int i, float hh) {
        hv[i & 3] = hh;
        if ((i & 3) != 3) return;
        const int g = i >> 2;
        const uint32_t y01 = pack_bf16x2(hv[0], hv[1]);
        const uint32_t y23 = pack_bf16x2(hv[2], hv[3]);
        // four tokens into the wave's patch: the low halves of the packed
        // pairs, and the high halves as they are
        const uint32_t pw = patch_w_lane + 4 * (g & 1) * kPatchStride;
        asm volatile(
            "ds_write_b16 %0, %1\n\t"
            "ds_write_b16_d16_hi %0, %1 offset:%3\n\t"
            "ds_write_b16 %0, %2 offset:%4\n\t"
            "ds_write_b16_d16_hi %0, %2 offset:%5"
            :
            : "v"(pw), "v"(y01), "v"(y23), "n"(kPatchStride),
              "n"(2 * kPatchStride), "n"(3 * kPatchStride)
            : "memory");
        if (g & 1) {
          // sixteen finished tokens are read back as 16-byte row chunks (the
          // LDS unit executes a wave's instructions in order)
          y_pending[g >> 1] = *reinterpret_cast<lds_u32x4*>(lds3 + patch_r_lane);
          asm volatile("" ::: "memory");
        }
      });
    }
    if (GELU) {
      // y * gelu(gate branch), each factor a bf16 tensor as in the reference:
      // the arithmetic and roundings of the stand-alone gelu_mul pass
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          y_pending[j][k] = gelu_mul_bf16x2(y_pending[j][k], g_pending[j][k]);
    }
    y_pending_row = (uint32_t)t_blk * row_bytes;
  };
  auto phase_g = [&](int kb, auto ODD) {
    constexpr bool odd = decltype(ODD)::value;
    if (!odd && team == 0) wait_vmcnt<2>();
    if (__builtin_expect(m_cur != 0 || (kb + 1) * kBT > T_len, 0))
      phase_g_as(kb, std::true_type{});
    else
      phase_g_as(kb, std::false_type{});
    if (odd) {
      m_prev = m_cur;
      m_cur = m_next;
      m_next = start_mask((kb >> 1) + 2);
    }
  };

  // ---- prologue -------------------------------------------------------------
  // Everything the first phases need is requested before anything waits: the
  // raw rows of the first two tiles, the positions of three tiles, then the
  // weights and the conv taps (one memory round trip after the other would
  // cost a launch of short chunks a tenth of its time).
#pragma unroll
  for (int j = 0; j < kRawLoadsPerWave; ++j) {
    dma_tile(tile_begin, j);
    dma_tile(tile_begin + 1, j);
  }
  uint32_t first_lo[3], first_hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    fetch_seg(tile_begin - 1 + k);
    first_lo[k] = seg_lo;
    first_hi[k] = seg_hi;
  }
  // ---- this wave's weights: 32 channels of the head, both gates ------------
  {
    const f32x4* src = reinterpret_cast<const f32x4*>(p.w_packed) +
                       ((int64_t)(h * 8 + wave) * 16 * 2) * 64 + lane;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 w[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) w[i] = src[(16 * half + i) * 64];
      asm volatile("" ::"v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]),
                   "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]),
                   "v"(w[10]), "v"(w[11]), "v"(w[12]), "v"(w[13]), "v"(w[14]),
                   "v"(w[15]));
#pragma unroll
      for (int i = 0; i < 16; ++i) set_weight_frag(16 * half + i, w[i]);
    }
  }

  // ---- conv table ---------------------------------------------------------
  if (tid < 128) {
    uint32_t u0 = 0, u1 = 0, u2 = 0, u3 = 0x3f803f80u, ub = 0;
    if (p.conv_w != nullptr) {
      const uint16_t* cw = (const uint16_t*)p.conv_w + h * kBW + tid * 2;
      u0 = *reinterpret_cast<const uint32_t*>(cw);
      u1 = *reinterpret_cast<const uint32_t*>(cw + W);
      u2 = *reinterpret_cast<const uint32_t*>(cw + 2 * W);
      u3 = *reinterpret_cast<const uint32_t*>(cw + 3 * W);
      ub = *reinterpret_cast<const uint32_t*>(
          (const uint16_t*)p.conv_b + h * kBW + tid * 2);
    }
    // w0 multiplies x[t-3], w3 multiplies x[t] (layers.py:514)
    const u32x4 t0 = {(u0 & 0xffffu) | (u1 << 16), (u2 & 0xffffu) | (u3 << 16),
                      (u0 >> 16) | (u1 & 0xffff0000u),
                      (u2 >> 16) | (u3 & 0xffff0000u)};
    const u32x4 t1 = {ub << 16, ub & 0xffff0000u, 0u, 0u};
    *reinterpret_cast<u32x4*>(lds_raw + kConvTabOff + tid * 32) = t0;
    *reinterpret_cast<u32x4*>(lds_raw + kConvTabOff + tid * 32 + 16) = t1;
  }

  seg_lo = first_lo[0]; seg_hi = first_hi[0];
  m_prev = start_mask(tile_begin - 1);
  seg_lo = first_lo[1]; seg_hi = first_hi[1];
  m_cur = start_mask(tile_begin);
  seg_lo = first_lo[2]; seg_hi = first_hi[2];
  m_next = start_mask(tile_begin + 1);
  wait_vmcnt<0>();
  __syncthreads();  // conv table, raw tiles
  {
    const u32x4 t0 = *reinterpret_cast<const u32x4*>(lds_raw + kConvTabOff +
                                                     conv_pair_of_lane * 32);
    const u32x2 t1 = *reinterpret_cast<const u32x2*>(lds_raw + kConvTabOff +
                                                     conv_pair_of_lane * 32 + 16);
    conv.w10[0] = t0[0]; conv.w32[0] = t0[1];
    conv.w10[1] = t0[2]; conv.w32[1] = t0[3];
    conv.bias[0] = __uint_as_float(t1[0]);
    conv.bias[1] = __uint_as_float(t1[1]);
  }
  {
    ConvRows cr;
    load_rows(2 * tile_begin, cr);
    conv_with_cuts(lds3, conv, cr, conv_cuts(2 * tile_begin, m_cur, m_prev), xc_row);
  }
  phase_barrier();

  const bool timed = p.timing != nullptr && blockIdx.x == 0 && blockIdx.y == 0;
  uint64_t clk0 = 0, tick0 = 0;
  if (timed) {
    clk0 = __builtin_readcyclecounter();
    tick0 = __builtin_amdgcn_s_memrealtime();
  }
  // team 1 runs one phase behind team 0
  if (team == 1) phase_barrier();
  // (whole tiles: a block past the end of the sequence is all identity, and
  // its stores fall outside the descriptor)
  for (int kb = 2 * tile_begin; kb < 2 * tile_end; kb += 2) {
    phase_m(kb, std::false_type{});
    phase_barrier();
    phase_g(kb, std::false_type{});
    phase_barrier();
    phase_m(kb + 1, std::true_type{});
    phase_barrier();
    phase_g(kb + 1, std::true_type{});
    phase_barrier();
  }
  if (team == 0) phase_barrier();
  if (timed) {
    const uint64_t clk1 = __builtin_readcyclecounter();
    const uint64_t tick1 = __builtin_amdgcn_s_memrealtime();
    if (tid == 0) {
      p.timing[0] = clk1 - clk0;
      p.timing[1] = tick1 - tick0;
    }
  }
  buffer_store_16(y_pending[0], ry, y_lane_bytes, y_pending_row);
  buffer_store_16(y_pending[1], ry, y_lane_bytes, y_pending_row + 8u * row_bytes);

  if (MODE == kChunkSummary) {
    // this chunk from a zero state: h_end = prod(a) * h_in + hc
    const auto sw = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(prod), __float_as_uint(prod), false, false);
    const float total = __uint_as_float(sw[0]) * __uint_as_float(sw[1]);
    if (!upper) {
      const int64_t at = ((int64_t)b * p.chunks + chunk) * W + ch;
      p.ws_p[at] = total;
      p.ws_h[at] = hc;
    }
    return;
  }
  if (MODE == kChunkHead) {
    // whatever came before the row is in hc already: a summary with a zero
    // product makes the replay take hc as the next chunk's start
    if (!upper) {
      const int64_t at = (int64_t)b * p.chunks * W + ch;
      p.ws_p[at] = 0.0f;
      p.ws_h[at] = hc;
    }
    return;
  }
  if (!last_chunk) return;
  if (p.h_last && !upper) p.h_last[(int64_t)b * W + ch] = hc;

  // Masked conv state: rows T-3..T-1 of x, each zeroed if a document starts in
  // a later position of the row; rows before the sequence start are zero.
  if (p.cache_out && tid < 128) {
    const uint32_t c = h * kBW + tid * 2;
    uint16_t* cache = (uint16_t*)p.cache_out + (int64_t)b * 3 * W + c;
    bool later_start = false;
#pragma unroll
    for (int kk = 2; kk >= 0; --kk) {
      const int t = T_len - 3 + kk;
      uint32_t v = 0;
      if (t >= 0 && !later_start)
        v = __builtin_amdgcn_raw_buffer_load_b32(rx, 2u * c,
                                                 (uint32_t)t * row_bytes, 0);
      *reinterpret_cast<uint32_t*>(cache + (int64_t)kk * W) = v;
      if (t >= 0 && is_doc_start(p.segpos, p.seg_kind, (int64_t)b * T_len + t))
        later_start = true;
    }
  }
}

enum PrefillPass { kPassWholeRows = 0, kPassFirst = 1, kPassReplay = 2 };

// blockIdx.x: (row, head); blockIdx.y: which chunk (kPassFirst: chunk 0 with
// its outputs beside the summaries of chunks 1 .. n-2; kPassReplay: chunks
// 1 .. n-1).
template <int PASS, bool GELU>
__global__ void __launch_bounds__(kThreads) block_prefill_teams_bf16_kernel(
    FusedArgs p) {
  if (PASS == kPassWholeRows) {
    prefill_teams_body<kWholeRow, GELU>(p, 0);
  } else if (PASS == kPassReplay) {
    prefill_teams_body<kChunkReplay, GELU>(p, (int)blockIdx.y + 1);
  } else if (blockIdx.y == 0) {
    prefill_teams_body<kChunkHead, GELU>(p, 0);
  } else {
    prefill_teams_body<kChunkSummary, false>(p, (int)blockIdx.y);
  }
}

template <int PASS, bool GELU>
hipError_t launch_teams_pass_as(const FusedArgs& a, int grid_y, hipStream_t s) {
  static OncePerDevice once;
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)block_prefill_teams_bf16_kernel<PASS, GELU>,
      kTeamsLdsBytes);
  if (e != hipSuccess) return e;
  block_prefill_teams_bf16_kernel<PASS, GELU>
      <<<dim3((unsigned)(a.B * a.H), (unsigned)grid_y), kThreads, kTeamsLdsBytes,
         s>>>(a);
  return hipGetLastError();
}

template <int PASS>
hipError_t launch_teams_pass(const FusedArgs& a, int grid_y, hipStream_t s) {
  if (a.gate_branch) return launch_teams_pass_as<PASS, true>(a, grid_y, s);
  return launch_teams_pass_as<PASS, false>(a, grid_y, s);
}

}  // namespace

hipError_t launch_block_prefill_teams_bf16(const FusedArgs& a, hipStream_t s) {
  const int64_t blocks = (int64_t)a.B * a.H;
  if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
  if (!a.w_packed) return hipErrorInvalidValue;
  if (a.chunks <= 1) return launch_teams_pass<kPassWholeRows>(a, 1, s);
  if (a.chunks < 3 || a.chunks > 65535) return hipErrorInvalidValue;
  hipError_t e = launch_teams_pass<kPassFirst>(a, a.chunks - 1, s);
  if (e != hipSuccess) return e;
  return launch_teams_pass<kPassReplay>(a, a.chunks - 1, s);
}

}  // namespace rg
