// 4-bit codes in matrix products as they are: what the two kernels for 2 .. 16 rows of activations share (held_gemm.h,
// q4g32_batch_list.hip).
#ifndef RELAX_AMD_CSRC_CODE_PRODUCTS_H_
#define RELAX_AMD_CSRC_CODE_PRODUCTS_H_

#include "wq_device.h"

namespace wq {

// 8 codes as an operand: fp16 numbers whose bits are the codes, that is 2^-24 (q0, q4), 2^-20 (q1, q5) and so on
__device__ __forceinline__ half8_t code_operand(uint32_t w) {
  const uint32_t w8 = w >> 8;
  return __builtin_bit_cast(half8_t, uint4_t{w & 0x000F000Fu, w & 0x00F000F0u, w8 & 0x000F000Fu, w8 & 0x00F000F0u});
}

// What a load has brought, in registers of its own: those of the load take the next one's.
__device__ __forceinline__ void take_words(const uint4_t& l, uint32_t (&w)[4]) {
  asm("v_mov_b32 %0, %4\n\tv_mov_b32 %1, %5\n\tv_mov_b32 %2, %6\n\tv_mov_b32 %3, %7\n\ts_nop 1"
      : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3])
      : "v"(l.x), "v"(l.y), "v"(l.z), "v"(l.w));
}

// Of two loads of 8 rows x 2 halves the two halves of both: lanes 8 .. 15 of every 16 take the first half from the second load 8
// lanes below, lanes 0 .. 7 the second half from the first load 8 lanes above (row_ror:8 turns a row of 16 lanes by 8).
__device__ __forceinline__ void exchange_halves(uint32_t (&a)[4], uint32_t (&b)[4]) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t lo = a[d], hi = b[d];
    a[d] = (uint32_t)__builtin_amdgcn_update_dpp((int)lo, (int)hi, 0x128 /* row_ror:8 */, 0xf, 0xc, false);
    b[d] = (uint32_t)__builtin_amdgcn_update_dpp((int)hi, (int)lo, 0x128, 0xf, 0x3, false);
  }
}

// a[g]: word kq of group g in lane quarter kq, from word g of group kq
__device__ __forceinline__ void spread_words(uint32_t (&a)[4]) {
  const auto h0 = __builtin_amdgcn_permlane32_swap(a[0], a[2], false, false);
  const auto h1 = __builtin_amdgcn_permlane32_swap(a[1], a[3], false, false);
  const auto q0 = __builtin_amdgcn_permlane16_swap(h0[0], h1[0], false, false);
  const auto q1 = __builtin_amdgcn_permlane16_swap(h0[1], h1[1], false, false);
  a[0] = q0[0], a[1] = q0[1], a[2] = q1[0], a[3] = q1[1];
}

// The operand's 16 rows hold up to 8 rows of activations at two halves of K, twice: lane (i, kq) of the products with columns
// 0 .. 7 (lo) and 8 .. 15 (hi) at the half i / 8 has rows 4 (kq mod 2) .. + 3 at half kq / 2, sums where the halves agree.
// They come together in the lanes with i < 8, quarters 0 and 1 for columns 0 .. 7, 2 and 3 for 8 .. 15.
__device__ __forceinline__ float join_halves(float lo, float hi) {
  const auto p = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi), false, false);
  const uint32_t mine = p[0], other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)p[1], 0x128 /* row_ror:8 */, 0xf, 0xf, false);
  return __builtin_bit_cast(float, mine) + __builtin_bit_cast(float, other);
}

}  // namespace wq
#endif  // RELAX_AMD_CSRC_CODE_PRODUCTS_H_
