// Gate weights of the bf16 prefill kernels with two waves per SIMD: resident
// in hand-numbered accumulation registers.
#ifndef RG_WEIGHT_FRAGS_H_
#define RG_WEIGHT_FRAGS_H_

#include "rg_common.h"

namespace rg {

// The wave's 32 weight fragments (fragment F = 2 k-step + gate, four registers
// each) live in the accumulation registers a[4F : 4F+3], written and read by
// inline assembly with the register numbers spelled out.
#define RG_TFRAG_CASES(X)                                                     \
  X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13)   \
  X(14) X(15) X(16) X(17) X(18) X(19) X(20) X(21) X(22) X(23) X(24) X(25)     \
  X(26) X(27) X(28) X(29) X(30) X(31)

__device__ __forceinline__ void set_weight_frag(int F, f32x4 v) {
  switch (F) {
#define RG_SET_CASE(F)                                                   \
  case F:                                                                \
    asm volatile("v_accvgpr_write_b32 a[" #F "*4], %0\n\t"               \
                 "v_accvgpr_write_b32 a[" #F "*4+1], %1\n\t"             \
                 "v_accvgpr_write_b32 a[" #F "*4+2], %2\n\t"             \
                 "v_accvgpr_write_b32 a[" #F "*4+3], %3"                  \
                 :                                                       \
                 : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3])            \
                 : "a127");                                              \
    break;
    RG_TFRAG_CASES(RG_SET_CASE)
#undef RG_SET_CASE
  }
}
__device__ __forceinline__ void mfma_weight_frag(int F, bool first,
                                                 const f32x4& a, f32x16& acc) {
  switch (F) {
#define RG_MFMA_CASE(F)                                                        \
  case F:                                                                      \
    if (first)                                                                 \
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, a[" #F "*4:" #F "*4+3], 0" \
                   : "=&v"(acc)                                                \
                   : "v"(a));                                                  \
    else                                                                       \
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, a[" #F "*4:" #F            \
                   "*4+3], %0"                                                 \
                   : "+v"(acc)                                                 \
                   : "v"(a));                                                  \
    break;
    RG_TFRAG_CASES(RG_MFMA_CASE)
#undef RG_MFMA_CASE
  }
}

}  // namespace rg
#endif  // RG_WEIGHT_FRAGS_H_
