// Whole recurrent core of a prefill in one launch (bf16, 256-wide heads) for
// numbers of (row, head) pairs that do not come out even on the CUs: blocks of 32
// tokens are dealt to workgroups as they ask for them, and the state of a row is
// handed from workgroup to workgroup through memory.
//
// A workgroup of eight waves belongs to one head, whose weights its waves keep in
// accumulation registers, and takes that head's blocks from a ticket counter:
// ticket j is block j / B of row j % B, so the rows advance side by side.  What a
// block goes through is rg_prefill_teams.hip's: two teams of waves one phase apart,
// phase M (matrix instructions, the conv of the next block) and phase G (gates,
// recurrence).  Between the gates and the outputs a block needs the state behind
// the block before it, which another workgroup has:
//   * a lane reduces its sixteen tokens to (prod a, state from zero), the halves of
//     the wave are joined, and as soon as the incoming state h is there the state
//     behind the block, P h + H, goes out to the next one: one multiply-add between
//     receiving and passing on.  Then the tokens are replayed from h;
//   * a state is one 8-byte word per channel: each of its halves has 16 bits of the
//     value and the 16 low bits of the block's number, written with an agent-scope
//     store of the whole word and polled by agent-scope loads into LDS, four bytes a
//     lane: a half vouches for itself, so it does not matter that two lanes fetch a
//     word; no fence, no flag apart.  (A load into a register on one of two paths, or
//     one for some lanes only, makes the compiler wait for loads and stores it need
//     not wait for.)  Two words per row and channel are enough: the word of block
//     t - 2 has been read when the state of block t - 1 arrives.
// Every wait ends: a workgroup takes tickets in order and works on them in order, a
// block waits only for a block of a smaller ticket (and its team's earlier phases),
// and a ticket is taken only by a workgroup that runs, however many of them do.
//
// What bounds it: as rg_prefill_teams.hip, at 9 to 13 % more a block (the summary and
// the hand-over, the four rows before every block read again), while there are rows
// enough; with few rows a head the way of a state from store to load (0.3 .. 0.6 us
// on an idle chip, 1.4 us a block of a row in all).  Blocks of 32 because the phases
// are; longer ones would hand over less often, but leave the last round less even.
// us before and after (rows or chunks by the workgroup / blocks): 2560 wide, joined,
// 8 x 4096 tokens 241 / 221, 12 x 4096 339 / 297, 26 x 1024 220 / 165, 26 x 4096
// 813 / 600; 4096 wide, 6 x 4096 joined 292 / 240, 20 x 4096 612 / 560, joined
// 815 / 723.
//
// Replaces the chain Conv1D.forward -> RGLRU.forward of
// recurrentgemma/torch/modules.py:632-643 (layers.py:447-529, 313-365, 140-191) for
// such shapes.
#include <type_traits>

#include "rg_common.h"
#include "rg_internal.h"
#include "rg_two_teams.h"

namespace rg {
namespace {

using namespace two_teams;

// Raw x of a block as the memory pipe writes it into LDS: rows -4 .. 31, 512 bytes
// each, two rows a load, three loads a wave (the six beyond 18 are sent out of
// range); a ring of three blocks.
constexpr int kRawLoads = (kBT + kRawHalo) / 2;
constexpr int kRawLoadsPerWave = (kRawLoads + kWaves - 1) / kWaves;
constexpr int kRawBlockBytes = kRawLoadsPerWave * kWaves * 2 * kRawRowBytes;
constexpr int kRing = kXcRing;

constexpr int kXcOff = 0;
constexpr int kRawOff = kXcOff + kRing * kXcBlockBytes;
constexpr int kPatchOff = kRawOff + kRing * kRawBlockBytes;
constexpr int kConvTabOff = kPatchOff + kWaves * kPatchBytesPerWave;
constexpr int kTicketOff = kConvTabOff + kConvTabBytes;  // the last eight tickets
// Per wave: the 32 state words that come into its block, as the memory pipe writes
// them, two polls of them; and the gate-branch values of its part of the block.
constexpr int kWordOff = kTicketOff + 8 * 4;
constexpr int kWordBytes = 32 * 8;
constexpr int kWordBytesPerWave = 2 * kWordBytes;
constexpr int kBranchOff = kWordOff + kWaves * kWordBytesPerWave;
constexpr int kBranchBytesPerWave = 2 * 1024;
constexpr int kRelayLdsBytes = kBranchOff + kWaves * kBranchBytesPerWave;
static_assert(kRelayLdsBytes <= 160 * 1024, "LDS of one CU");
constexpr int kAgentScope = 16;  // sc1 of a buffer instruction (gfx950)

// GELU: y is written as y * gelu(gate_branch), the join of the recurrent block's two
// branches (recurrentgemma/torch/modules.py:627-628, 644).
template <bool GELU>
__global__ void __launch_bounds__(kThreads)
block_prefill_relay_bf16_kernel(FusedArgs p, int per_head, uint32_t inverse) {
  constexpr int kTailX = GELU ? kTailXJoined : kTailXPlain;
  constexpr int kTailA = GELU ? kTailAJoined : kTailAPlain;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  lds_byte* const lds3 = (lds_byte*)lds_raw;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int team = wave >> 2;
  const int in_team = wave & 3;
  // Workgroups go to the eight XCDs in turn: those of a head, which hand each other
  // states and read neighbouring rows of x, to one of them as far as that goes.
  int id = blockIdx.x;
  {
    const int per_xcd = (int)gridDim.x / 8;
    if (id < 8 * per_xcd) id = (id & 7) * per_xcd + (id >> 3);
  }
  const int h = id / per_head;
  const int T_len = p.T;
  const int64_t W = p.W;
  const int blocks = (T_len + kBT - 1) / kBT;  // of a row
  const int total = blocks * p.B;              // of this head (launcher: < 2^30)
  const bool upper = lane >= 32;
  const int n0 = wave * 32;  // first channel of this wave in the head
  const uint32_t row_bytes = 2u * (uint32_t)p.W;
  const uint32_t seq_bytes = (uint32_t)T_len * row_bytes;  // < 2^31 (launcher)
  const bool seg_is64 = p.seg_kind == kSegI64;
  const uint32_t seg_esize = seg_is64 ? 8u : 4u;

  // A ticket as a place: block t of row b; none beyond the last.
  struct Place {
    int b, t;
    bool any;
  };
  // (scalar arithmetic: inverse = (2^32 - 1) / B gives the quotient or one less)
  auto place_of = [&](int ticket) {
    Place q;
    q.any = ticket < total;
    const uint32_t j = q.any ? (uint32_t)ticket : 0u;
    uint32_t t = (uint32_t)(((uint64_t)j * inverse) >> 32);
    uint32_t b = j - t * (uint32_t)p.B;
    t += b >= (uint32_t)p.B ? 1u : 0u;
    b -= b >= (uint32_t)p.B ? (uint32_t)p.B : 0u;
    q.t = (int)t;
    q.b = (int)b;
    return q;
  };
  auto ticket_slot = [&](int k) {
    return reinterpret_cast<lds_u32*>(lds3 + kTicketOff + 4 * (k & 7));
  };
  auto place_at = [&](int k) {  // of this workgroup's k-th ticket
    return place_of((int)__builtin_amdgcn_readfirstlane(*ticket_slot(k)));
  };
  int* const counter = p.relay_tickets + h;
  auto take = [&]() { return atomicAdd(counter, 1); };

  // Positions of tokens t0 - 32 .. t0 + 31 of a block, one per lane; bit 32 + i of
  // the mask: token i starts a document.
  uint32_t seg_lo = 1, seg_hi = 0;
  bool seg_in = false;
  // (No branches here or in dma_block: they run between the matrix instructions.
  // Places beyond the last have descriptors of no bytes.)
  const uint32_t seg_hi_off = seg_is64 ? 4u : kBufferOutOfRange;
  auto fetch_seg = [&](const Place& q) {
    const __amdgpu_buffer_rsrc_t rseg =
        make_rsrc((const char*)p.segpos + (int64_t)q.b * T_len * seg_esize,
                  q.any ? (uint32_t)T_len * seg_esize : 0u);
    const int t = q.t * kBT + lane - 32;
    seg_in = (uint32_t)t < (q.any ? (uint32_t)T_len : 0u);
    const uint32_t off = (uint32_t)t * seg_esize;
    seg_lo = __builtin_amdgcn_raw_buffer_load_b32(rseg, off, 0, 0);
    seg_hi = __builtin_amdgcn_raw_buffer_load_b32(rseg, off + seg_hi_off, 0, 0);
  };
  auto start_mask = [&]() -> uint64_t {
    uint32_t lo = seg_lo, hi = seg_hi;
    asm volatile("" : "+v"(lo), "+v"(hi));
    return __ballot(seg_in && (lo | hi) == 0u);
  };

  const uint32_t dma_lane_off = 2u * (uint32_t)(h * kBW) +
                                16u * (uint32_t)(lane & 31) +
                                (uint32_t)(lane >> 5) * row_bytes;
  // this wave's load j of a block's raw rows
  auto dma_block = [&](const Place& q, int k, int j) {
    const int i = wave + kWaves * j;
    const __amdgpu_buffer_rsrc_t rx =
        make_rsrc((const char*)p.x + (int64_t)q.b * seq_bytes,
                  q.any && i < kRawLoads ? seq_bytes : 0u);
    const uint32_t voff = (uint32_t)((q.t * kBT - kRawHalo + 2 * i) *
                                     (int)row_bytes) + dma_lane_off;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rx, lds3 + kRawOff + (k % kRing) * kRawBlockBytes + i * 1024, 16, voff, 0,
        0, 0);
  };

  // ---- lane-dependent LDS offsets -------------------------------------------
  // conv: thread -> (channel pair tid % 128, rows 8 rg4 .. 8 rg4 + 7); the conv rows
  // in the order that gives a lane sixteen tokens in a row (rg_prefill_teams.hip)
  const int rg4 = team * 2 + (in_team >> 1);  // 0..3
  const int conv_pair_of_lane = (in_team & 1) * 64 + lane;
  const uint32_t conv_raw_lane =
      kRawOff + (uint32_t)(rg4 * kConvRows + kRawHalo - 3) * kRawRowBytes +
      conv_pair_of_lane * 4;
  const uint32_t conv_xc_lane =
      kXcOff + (uint32_t)(16 * (rg4 & 1) + 4 * (rg4 >> 1)) * kXcRowBytes +
      conv_pair_of_lane * 4;
  auto xc_row = [](int i) { return 8 * (i >> 2) + (i & 3); };
  // gates: lane -> channel n0 + lane % 32, tokens 16 (lane / 32) + ...
  const uint32_t xc_lane = kXcOff + 4u * (lane >> 5) * kXcRowBytes +
                           2u * (uint32_t)(n0 + (lane & 31));
  const uint32_t a_lane =
      kXcOff + (uint32_t)(lane & 31) * kXcRowBytes + 16u * (lane >> 5);
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
    conv_load(lds3, conv_raw_lane + (uint32_t)(kb % kRing) * kRawBlockBytes,
              conv_xc_lane + (uint32_t)(kb % kRing) * kXcBlockBytes, cr);
  };
  // Document starts among this thread group's rows (3 before + its own) of the block
  // with this mask
  auto conv_cuts = [&](uint64_t mask) -> uint32_t {
    return (uint32_t)(mask >> (29 + rg4 * kConvRows)) &
           ((1u << (kConvRows + 3)) - 1u);
  };

  // ---- state ------------------------------------------------------------------
  const int ch = h * kBW + n0 + (lane & 31);  // this lane's channel
  const float bias_x = -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[0])[ch]);
  const float bias_a = -kLog2e * bf16_bits_to_f32(((const uint16_t*)p.b[1])[ch]);
  const float inv_decay = inverse_decay(
      (-8.0f * kLog2e) *
      softplus_precise(bf16_bits_to_f32(((const uint16_t*)p.a_param)[ch])));
  f32x16 acc_x, acc_a;
  // conv outputs of the block in phase G, this lane's tokens, as floats
  uint32_t xr[16];
  u32x4 y_pending[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  int y_row = 0;  // where they belong
  uint32_t y_pending_row = kBufferOutOfRange;
  // states between blocks: [B][2][W] words.  Block t leaves its number + 1 in both
  // halves, mod 2^16: what it replaces has t - 1 there, or the zeros from before the
  // first two blocks
  // (lane-dependent addresses of phase G are made where they are used, out of the
  // compiler's sight: kept across phase M they are registers too many)
  auto lane_channel = [&]() {
    uint32_t c = (uint32_t)lane & 31u;
    asm volatile("" : "+v"(c));
    return c;
  };
  auto word_at = [&](int b, int t) {
    return p.relay_words + ((int64_t)b * 2 + (t & 1)) * W + h * kBW + n0 +
           lane_channel();
  };
  auto word_of = [](float value, int t) {
    const uint32_t v = __float_as_uint(value), number = (uint32_t)(t + 1) & 0xffffu;
    return (uint64_t)(v << 16 | number) << 32 | (v & 0xffff0000u) | number;
  };
  // the words that come into a block, into LDS (four bytes a lane)
  auto fetch_words = [&](const Place& q, int slot) {
    const __amdgpu_buffer_rsrc_t r = make_rsrc(
        p.relay_words + ((int64_t)q.b * 2 + ((q.t + 1) & 1)) * W + h * kBW + n0,
        q.t > 0 ? (uint32_t)kWordBytes : 0u);
    uint32_t off = 4u * (uint32_t)lane;
    asm volatile("" : "+v"(off));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        r, lds3 + kWordOff + wave * kWordBytesPerWave + slot * kWordBytes, 4, off, 0,
        0, kAgentScope);
  };
  // the gate-branch values at the positions of a block's outputs, into LDS
  lds_byte* const branch = lds3 + kBranchOff + wave * kBranchBytesPerWave;
  auto fetch_branch = [&](const Place& q) {
    const __amdgpu_buffer_rsrc_t r = make_rsrc(
        (const char*)p.gate_branch + (int64_t)q.b * seq_bytes, seq_bytes);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r, branch + 1024 * j, 16,
          y_lane_bytes + (uint32_t)(q.t * kBT + 8 * j) * row_bytes, 0, 0, 0);
  };
  auto state_row = [&](const float* base, int b) {
    return make_rsrc(base + (int64_t)b * W + h * kBW + n0, base ? 128u : 0u);
  };

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
  auto store_pending = [&]() {
    const __amdgpu_buffer_rsrc_t ry =
        make_rsrc((char*)p.y + (int64_t)y_row * seq_bytes, seq_bytes);
    buffer_store_16(y_pending[0], ry, y_lane_bytes, y_pending_row);
    buffer_store_16(y_pending[1], ry, y_lane_bytes,
                    y_pending_row + 8u * row_bytes);
  };

  // ---- phase M of the workgroup's block k: matrix instructions, y of the block
  //      before, conv of the next (mask: its document starts), rows and positions
  //      of the third after it; gives the starts of the second -------------------
  auto phase_m = [&](int k, uint64_t mask_next, const Place& first,
                     const Place& third) {
    uint64_t mask_second = 0;
    // The raw rows a wave asks for in one phase M are first read two phases after its
    // next one.  Team 1 has waited for them here (behind them it has issued two loads
    // of positions and no more than one store), team 0 at the top of phase G.
    if (team == 1) wait_vmcnt<2>();
    fetch_words(first, 0);
    __builtin_amdgcn_sched_barrier(0);  // (phase G counts what follows)
    if (GELU) fetch_branch(first);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t a_at = a_lane + (uint32_t)(k % kRing) * kXcBlockBytes;
    auto a_read = [&](int ks) {
      return *reinterpret_cast<lds_f32x4*>(lds3 + a_at + ks * 32);
    };
    f32x4 a[kARing];
#pragma unroll
    for (int q = 0; q < kARing - 1; ++q) a[q] = a_read(q);
    store_pending();
    const uint32_t cuts = conv_cuts(mask_next);
    ConvRows cr;
    const uint32_t x_at = xc_lane + (uint32_t)(k % kRing) * kXcBlockBytes;
#define RG_XR(i)                                                            \
  asm volatile("v_mov_b32 %0, 0\n\tds_read_u16_d16_hi %0, %1 offset:%2"      \
               : "=&v"(xr[i])                                                \
               : "v"(x_at), "n"((8 * ((i) >> 2) + ((i) & 3)) * kXcRowBytes));
    __builtin_amdgcn_s_setprio(kMatrixPriority);
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
      if (ks + kARing - 1 < 16)
        a[(ks + kARing - 1) % kARing] = a_read(ks + kARing - 1);
      mfma_weight_frag(2 * ks, ks == 0, a[ks % kARing], acc_x);
      mfma_weight_frag(2 * ks + 1, ks == 0, a[ks % kARing], acc_a);
      if (ks == 0) load_rows(k + 1, cr);
      if (ks >= 3 && ks % 3 == 0 && ks / 3 - 1 < kConvRows / 2)
        conv_pair(lds3, conv, cr, ks / 3 - 1, xc_row);
      if (ks == 1) dma_block(third, k + 3, 0);
      if (ks == 2) dma_block(third, k + 3, 1);
      if (ks == 3) dma_block(third, k + 3, 2);
      if (ks == 13) { RG_XR(0) RG_XR(1) RG_XR(2) RG_XR(3) RG_XR(4) }
      if (ks == 14) { RG_XR(5) RG_XR(6) RG_XR(7) RG_XR(8) RG_XR(9) RG_XR(10) }
      if (ks == 15) { RG_XR(11) RG_XR(12) RG_XR(13) RG_XR(14) RG_XR(15) }
      if (ks == 15) {
        mask_second = start_mask();
        fetch_seg(third);
      }
    }
#undef RG_XR
    __builtin_amdgcn_s_setprio(0);
    if (__builtin_expect(cuts != 0, 0)) conv_with_cuts(lds3, conv, cr, cuts, xc_row);
    // the last matrix results land (19 issue slots); every reader of the
    // accumulators is ordered behind this statement
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc_x), "+v"(acc_a));
    gate_x(0, kTailX);
    gate_a(0, kTailA);
    // (computed here, before the barrier: nothing else orders them)
    asm volatile("" : "+v"(acc_x), "+v"(acc_a));
    return mask_second;
  };

  // ---- phase G of a block ------------------------------------------------------
  auto phase_g_as = [&](const Place& q, uint32_t block_starts, auto GENERAL) {
    constexpr bool general = decltype(GENERAL)::value;
    const int t_blk = q.t * kBT;
    // The words asked for in phase M (behind them that phase issued seven loads and
    // stores, with the join nine): where the block before was not done by then, asked
    // for again now and behind the gates, and then until it is, two polls in flight.
    // (All of it by way of LDS: a load into registers on one of two paths makes the
    // compiler wait for everything on both.)
    uint32_t state = 0;
    auto arrived = [&](int slot) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const uint64_t word =
          *reinterpret_cast<lds_u64*>(lds3 + kWordOff + wave * kWordBytesPerWave +
                                      slot * kWordBytes + 8 * lane_channel());
      const uint32_t low = (uint32_t)word, high = (uint32_t)(word >> 32);
      state = __builtin_amdgcn_perm(low, high, 0x07060302u);
      // both halves from the block before
      return (bool)__all(__builtin_amdgcn_perm(low, high, 0x05040100u) ==
                         ((uint32_t)q.t & 0xffffu) * 0x10001u);
    };
    wait_vmcnt<GELU ? 9 : 7>();
    bool there = q.t == 0 || arrived(0);
    if (!there) fetch_words(q, 0);
    __builtin_amdgcn_sched_barrier(0);
    gate_x(kTailX, 16);
    gate_a(kTailA, 16);
    float xn[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) xn[i] = __uint_as_float(xr[i]) * acc_x[i];
    if (general) {
      // document start: a = 0; past the end of the sequence: a = 1, no input.
      // The input scale sqrt(1 - a^2) comes out as 1 at a start.
      int first = (lane >> 5) * 16;
      asm volatile("" : "+v"(first));
      const uint32_t starts = block_starts >> first;
      const int left = T_len - t_blk - first;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        acc_a[i] = ((starts >> i) & 1u) ? 0.0f : acc_a[i];
        acc_a[i] = i < left ? acc_a[i] : 1.0f;
        xn[i] = i < left ? xn[i] : 0.0f;
      }
    }
    // the half block as (prod a, state from zero), the halves joined
    float e1 = 0.0f, p1 = 1.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      xn[i] = xn[i] *
              __builtin_amdgcn_sqrtf(__builtin_fmaf(-acc_a[i], acc_a[i], 1.0f));
      e1 = __builtin_fmaf(acc_a[i], e1, xn[i]);
      p1 *= acc_a[i];
    }
    const auto se = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(e1), __float_as_uint(e1), false, false);
    const auto sp = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(p1), __float_as_uint(p1), false, false);
    const float e_low = __uint_as_float(se[0]), p_low = __uint_as_float(sp[0]);
    const float e_up = __uint_as_float(se[1]), p_up = __uint_as_float(sp[1]);
    if (!there) {
      fetch_words(q, 1);
      for (int polls = 0; ; ++polls) {
        wait_vmcnt<1>();
        if (arrived(polls & 1)) break;
        if (polls == kMaxStatePolls) {
          state = kNoState;
          break;
        }
        fetch_words(q, polls & 1);
      }
    }
    float h_in = __uint_as_float(state);
    if (q.t == 0)
      h_in = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          state_row(p.h0, q.b), 4u * lane_channel(), 0, 0));
    // state behind the lower half, behind the block: passed on at once
    const float h_mid = __builtin_fmaf(p_low, h_in, e_low);
    const float h_out = __builtin_fmaf(p_up, h_mid, e_up);
    if (!upper) {
      if (q.t + 1 < blocks)
        __hip_atomic_store(word_at(q.b, q.t), word_of(h_out, q.t), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      else  // (no descriptor, no store)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(h_out),
                                              state_row(p.h_last, q.b),
                                              4u * lane_channel(), 0, 0);
    }
    float hh = upper ? h_mid : h_in;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float hv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        hh = __builtin_fmaf(acc_a[4 * g + i], hh, xn[4 * g + i]);
        hv[i] = hh;
      }
      const uint32_t y01 = pack_bf16x2(hv[0], hv[1]);
      const uint32_t y23 = pack_bf16x2(hv[2], hv[3]);
      asm volatile(
          "ds_write_b16 %0, %1 offset:%3\n\t"
          "ds_write_b16_d16_hi %0, %1 offset:%4\n\t"
          "ds_write_b16 %0, %2 offset:%5\n\t"
          "ds_write_b16_d16_hi %0, %2 offset:%6"
          :
          : "v"(patch_w_lane), "v"(y01), "v"(y23),
            "n"((4 * (g & 1)) * kPatchStride),
            "n"((4 * (g & 1) + 1) * kPatchStride),
            "n"((4 * (g & 1) + 2) * kPatchStride),
            "n"((4 * (g & 1) + 3) * kPatchStride)
          : "memory");
      if (g & 1) {
        // sixteen finished tokens are read back as 16-byte row chunks (the LDS
        // unit executes a wave's instructions in order)
        y_pending[g >> 1] = *reinterpret_cast<lds_u32x4*>(lds3 + patch_r_lane);
        asm volatile("" ::: "memory");
      }
    }
    if (GELU) {
      wait_vmcnt<7>();  // (the branch, asked for in phase M before seven others)
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const u32x4 g = *reinterpret_cast<lds_u32x4*>(branch + 1024 * j + 16 * lane);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          y_pending[j][i] = gelu_mul_bf16x2(y_pending[j][i], g[i]);
      }
    }
    y_row = q.b;
    y_pending_row = (uint32_t)t_blk * row_bytes;
  };

  // ---- prologue -------------------------------------------------------------
  // The weights' way from memory and the first tickets' run side by side.
  {
    const f32x4* src = reinterpret_cast<const f32x4*>(p.w_packed) +
                       ((int64_t)(h * 8 + wave) * 16 * 2) * 64 + lane;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 w[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) w[i] = src[(16 * half + i) * 64];
      if (tid == 0) {
#pragma unroll
        for (int i = 0; i < 3 - half; ++i)
          *ticket_slot(3 * half + i) = (uint32_t)take();
      }
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

  __syncthreads();  // conv table, tickets
  Place now = place_at(0), next = place_at(1);
#pragma unroll
  for (int j = 0; j < kRawLoadsPerWave; ++j) dma_block(now, 0, j);
#pragma unroll
  for (int j = 0; j < kRawLoadsPerWave; ++j) dma_block(next, 1, j);
  Place second = place_at(2);
#pragma unroll
  for (int j = 0; j < kRawLoadsPerWave; ++j) dma_block(second, 2, j);
  fetch_seg(now);
  uint64_t mask_now = start_mask();
  fetch_seg(next);
  uint64_t mask_next = start_mask();
  fetch_seg(second);
  wait_vmcnt<0>();
  __syncthreads();  // raw rows
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
    load_rows(0, cr);
    conv_with_cuts(lds3, conv, cr, conv_cuts(mask_now), xc_row);
  }
  phase_barrier();

  // team 1 runs one phase behind team 0
  if (team == 1) phase_barrier();
  int asked = 0;
  for (int k = 0; now.any; ++k) {
    // team 0's first wave asks for the fifth ticket from here on, and lays what it
    // asked for a block ago into LDS (there by now, and read a block from here)
    if (wave == 0 && lane == 0) {
      if (k > 0) *ticket_slot(k + 4) = (uint32_t)asked;
      asked = take();
    }
    const Place third = place_at(k + 3);
    const uint64_t mask_second = phase_m(k, mask_next, now, third);
    phase_barrier();
    const uint32_t starts = (uint32_t)(mask_now >> 32);
    if (__builtin_expect(starts != 0 || (now.t + 1) * kBT > T_len, 0))
      phase_g_as(now, starts, std::true_type{});
    else
      phase_g_as(now, starts, std::false_type{});
    phase_barrier();
    mask_now = mask_next;
    mask_next = mask_second;
    now = next;
    next = second;
    second = third;
  }
  if (team == 0) phase_barrier();
  store_pending();
}

// Before the other kernel: no state word valid, no ticket taken; and the conv state,
// rows T-3..T-1 of x, each zeroed if a document starts in a later position of the
// row; rows before the sequence start are zero.
__global__ void __launch_bounds__(256) relay_begin_kernel(FusedArgs p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t W = p.W;
  if (i < p.H) p.relay_tickets[i] = 0;
  if (i >= (int64_t)p.B * W / 2) return;  // two channels of a row each
  const int b = (int)(2 * i / W);
  const int64_t c = 2 * i - b * W;
#pragma unroll
  for (int s = 0; s < 2; ++s)
    *reinterpret_cast<u32x4*>(p.relay_words + ((int64_t)b * 2 + s) * W + c) =
        u32x4{0, 0, 0, 0};
  if (!p.cache_out) return;
  uint16_t* const cache = (uint16_t*)p.cache_out + (int64_t)b * 3 * W + c;
  bool later_start = false;
#pragma unroll
  for (int kk = 2; kk >= 0; --kk) {
    const int t = p.T - 3 + kk;
    uint32_t v = 0;
    if (t >= 0 && !later_start)
      v = *reinterpret_cast<const uint32_t*>((const uint16_t*)p.x +
                                             ((int64_t)b * p.T + t) * W + c);
    *reinterpret_cast<uint32_t*>(cache + (int64_t)kk * W) = v;
    if (t >= 0 && is_doc_start(p.segpos, p.seg_kind, (int64_t)b * p.T + t))
      later_start = true;
  }
}

template <bool GELU>
hipError_t launch_as(const FusedArgs& a, int per_head, hipStream_t s) {
  static OncePerDevice once;
  hipError_t e = set_max_dynamic_lds(
      once, (const void*)block_prefill_relay_bf16_kernel<GELU>, kRelayLdsBytes);
  if (e != hipSuccess) return e;
  block_prefill_relay_bf16_kernel<GELU>
      <<<dim3((unsigned)(per_head * a.H)), kThreads, kRelayLdsBytes, s>>>(
          a, per_head, 0xffffffffu / (uint32_t)a.B);
  return hipGetLastError();
}

}  // namespace

// Against rows by the workgroup (rg_prefill_teams.hip) and rows in chunks
// (rg_prefill.hip), in us as measured at 8, 10 and 16 heads, 1 to 64 rows of 256 to
// 4096 tokens, and at 70 other shapes of 3 to 32 heads: what it sends here is at most
// 2 % slower here and up to 35 % faster (apart / here: joined, 2560 wide, 26 rows of
// 1024 220 / 165, 28 of 500 117 / 96, 52 of 2048 632 / 593; 4096 wide, 4 of 2048
// 112 / 95, 10 of 2650 269 / 250; not joined, 20 of 4096 612 / 560).  What it keeps
// apart: pairs that come out even (4096 wide, 16 of 4096 joined 513 / 577, 32 of 1024
// 276 / 306), short rows (2560 wide, 24 of 512 65 / 87), few pairs (2560 wide, 2 of
// 4096 86 / 117), whose states go from hand to hand more slowly than chunks are
// joined.
bool prefill_relay_pays(int B, int H, int T, bool joined) {
  if (B <= 0 || H <= 0 || H > 256 || T < 384 ||
      ((int64_t)T + kBT - 1) / kBT * B > (1 << 30))
    return false;
  const float pairs = (float)B * (float)H;
  const float tiles = (float)((T + 63) / 64);
  // here: by the work of a workgroup, at least by the steps of a row
  const float rows = (float)B / (float)(256 / H);  // of a workgroup
  const float step = joined ? 8.7f : 6.75f;
  const float here = 21.0f + tiles * fmaxf(step * rows, joined ? 2.9f : 2.4f);
  const float round = (joined ? 7.9f : 6.05f) * tiles + (joined ? 7.0f : 3.0f);
  float apart;
  if (pairs > 256.0f) {
    // whole rounds, and a last one that takes 0.58 of a round's time however few
    // pairs are in it
    const float whole = floorf(pairs / 256.0f);
    const float last = pairs / 256.0f - whole;
    apart = round * (whole + (last > 0.0f ? fmaxf(0.58f, 0.37f + 0.6f * last) : 0.0f));
  } else if (pairs > 128.0f) {
    apart = round * (0.44f + 0.56f / 256.0f * pairs);
  } else {
    return T >= 1000 && pairs >= (joined ? 40.0f : T >= 2000 ? 60.0f : 90.0f);
  }
  return here < 0.97f * apart;
}

size_t prefill_relay_workspace_bytes(int B, int W, int H) {
  return (size_t)B * 2 * W * sizeof(uint64_t) + (((size_t)H * 4 + 15) & ~(size_t)15);
}

hipError_t launch_block_prefill_relay_bf16(FusedArgs a, void* workspace,
                                           hipStream_t s) {
  const int64_t blocks = ((int64_t)a.T + kBT - 1) / kBT * a.B;
  if (!a.w_packed || !workspace || a.B <= 0 || a.H <= 0 || a.H > 256 ||
      a.W != a.H * kBW || blocks <= 0 || blocks > (1 << 30) ||
      (int64_t)a.T * a.W * 2 >= (int64_t)0x7fffffff)
    return hipErrorInvalidValue;
  a.relay_words = (uint64_t*)workspace;
  a.relay_tickets = (int*)(a.relay_words + (size_t)a.B * 2 * a.W);
  const int64_t items = (int64_t)a.B * a.W / 2;  // (at least H)
  relay_begin_kernel<<<dim3((unsigned)((items + 255) / 256)), 256, 0, s>>>(a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  int per_head = 256 / a.H;
  if (per_head > blocks) per_head = (int)blocks;
  return a.gate_branch ? launch_as<true>(a, per_head, s)
                       : launch_as<false>(a, per_head, s);
}

}  // namespace rg
