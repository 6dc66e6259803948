// What the kernels share that number their accumulation registers by hand and bring
// their operands to LDS by the memory pipe in inline assembly (rg_matmul.hip,
// rg_attention_prefill.hip).
#ifndef RG_MATRIX_ASM_H_
#define RG_MATRIX_ASM_H_

#include <utility>

#include "rg_common.h"

namespace rg {
namespace matrix_asm {

typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

template <int... I, class F>
__device__ __forceinline__ void for_each(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_n(F&& f) {
  for_each(std::make_integer_sequence<int, N>{}, f);
}

// ------------------------------------------------------- accumulators ----
// Blocks of 16 x 16 results in a[0:255], four registers each.  The build checks that
// the compiler allocates none of them for itself.
__device__ __forceinline__ void take_accumulators() { asm volatile("" ::: "a255"); }
template <int N>
__device__ __forceinline__ float acc_read() {
  float t;
  asm volatile("v_accvgpr_read_b32 %0, a[%c1]" : "=v"(t) : "n"(N));
  return t;
}
template <int N>
__device__ __forceinline__ void acc_write(float t) {
  asm volatile("v_accvgpr_write_b32 a[%c1], %0" ::"v"(t), "n"(N));
}
template <int N>
__device__ __forceinline__ void acc_zero() {
  asm volatile("v_accvgpr_write_b32 a[%c0], 0" ::"n"(N));
}
// block BLK += a x b
template <int BLK>
__device__ __forceinline__ void acc_mfma(const f32x4& a, const f32x4& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 a[%c2:%c2+3], %0, %1, a[%c2:%c2+3]" ::"v"(a),
               "v"(b), "n"(4 * BLK));
}
// The compiler does not count the wait states between a matrix instruction in inline
// assembly and a read of its result.
__device__ __forceinline__ void wait_for_matrix_results() {
  asm volatile("s_nop 15\n\ts_nop 7");
}

// -------------------------------------------------------- loads to LDS ----
// (inline assembly: behind the builtin the compiler has every transposing LDS read wait
// for all loads on their way)

// A buffer descriptor in scalar registers.
__device__ __forceinline__ u32x4 scalar_rsrc(const void* base, int64_t bytes) {
  const uint64_t at = (uint64_t)base;
  return u32x4{
      (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at),
      (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32)) & 0xffffu,
      (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

// 16 bytes a lane, lane after lane, to LDS bytes to + OFFSET ..: of `rsrc` at byte
// v + at.  What lies behind the descriptor's end is zero, also where the scalar offset
// alone does (tried with scalar offsets of 0 to 128 times the descriptor's size, in a
// buffer that held them all).  M0, which says where to, is read one wait state behind its
// write at the earliest: the compiler, which writes M0 for the builtin, puts an instruction
// between, and the build fails where one of these has none (check_mfma_wait.py).  (Nothing
// else in the kernels that use these reads M0.)
template <int OFFSET>
__device__ __forceinline__ void load_lds_16(uint32_t to, uint32_t v, u32x4 rsrc, int at) {
  asm volatile(
      "s_add_u32 m0, %0, %c1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds" ::"s"(to),
      "n"(OFFSET), "v"(v), "s"(rsrc), "s"(at)
      : "scc");
}
// The same with four bytes a lane.
__device__ __forceinline__ void load_lds_4(uint32_t to, uint32_t v, u32x4 rsrc) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(to),
               "v"(v), "s"(rsrc));
}

}  // namespace matrix_asm
}  // namespace rg

#endif  // RG_MATRIX_ASM_H_
