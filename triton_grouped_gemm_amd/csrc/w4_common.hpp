// Building blocks shared by the four-wave gfx950 kernels (gemm_w4.hip, gemm_wgrad.hip): multiplies and fragment reads as
// single inline-assembly statements, which the compiler keeps in source order and only allocates registers for.
#pragma once
#include "fast_common.hpp"

namespace tgg {

template <int DT> TGG_DEV void mfma_acc(f32x4_t& acc, const i32x4_t& w, const i32x4_t& x) {
  if (DT == DT_BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
}

// The same with a zero addend: the first K step of a tile starts its accumulators afresh
template <int DT> TGG_DEV void mfma_new(f32x4_t& acc, const i32x4_t& w, const i32x4_t& x) {
  if (DT == DT_BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(w), "v"(x));
}

// 16-byte fragment of a K-contiguous operand
template <int OFF> TGG_DEV void lds_read_b128(i32x4_t& dst, uint32_t addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF) : "memory");
}
// fragment of a token-row operand: two transposing 8-byte reads (K 0..3 and 4..7 of the lane's column)
template <int OFF0, int OFF1> TGG_DEV void lds_read_tr(i32x4_t& dst, uint32_t addr) {
  i32x2_t lo, hi;
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
               : "=&v"(lo), "=&v"(hi) : "v"(addr), "n"(OFF0), "n"(OFF1) : "memory");
  dst = __builtin_shufflevector(lo, hi, 0, 1, 2, 3);
}
#define TGG_TIE8(f) "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7])

}  // namespace tgg
