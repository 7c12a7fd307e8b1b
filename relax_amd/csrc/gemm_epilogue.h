// Row-wise epilogue shared by the MFMA GEMM kernels.
//
// After v_mfma_f32_32x32x16_f16 accumulator register r of lane (j, h) is element
// (row 8*(r/4) + 4*h + r%4, col j) of its 32x32 sub-tile: a lane holds single columns, so
// direct stores would be 2-byte accesses in 64-byte runs.  Instead each wavefront transposes
// the fp32 accumulators through its own piece of LDS, one row sub-tile at a time, and then
// handles 8 consecutive columns of a row per lane: bias / residual reads and the store are 16 bytes
// wide.  They are typed with the alignment of a half: the hardware takes 16-byte accesses at any 2-byte
// address, so odd N and unaligned operands use the same instructions (q4f16_1, N = 4097, K = 4096, M = 2048:
// 105 -> 94 us, with a residual at M = 512 56 -> 39 us); the last columns of a row where N % 8 != 0 go one by one.
//
// An Epilogue provides
//   half_t  operator()(float acc, int m, int n)                 one element
//   half8_t apply8(const float (&v)[8], int m, int n)           columns n .. n+7 of row m
// and, only where an element costs far more than its share of a row pass (erf, exp),
//   bool    activates()            the staged values take activate() first, apply8 then sees its results
//   float   column_bias(int n)     what activate() needs of column n, loaded once per lane and tile
//   float   activate(float acc, float column_bias, int m, int n)
//                                  (the columns of such a format come in eights: its rows have no tail)
// That pass is a rolled loop over LDS: inlined next to each of the 64 .. 256 accumulators of a lane it was
// megabytes of code, and eight at a time spilled.  With it 256 x 256 tiles can take these calls, which is most of the gain
// (int8, K = 8192, N = 28672, M = 500, with the branch-free erf of wq_device.h: gelu 339 -> 249 us, silu 316 -> 251 us,
// bias alone 234 us).
#ifndef RELAX_AMD_CSRC_GEMM_EPILOGUE_H_
#define RELAX_AMD_CSRC_GEMM_EPILOGUE_H_

#include <type_traits>

#include "wq_device.h"

namespace wq {

typedef _Float16 half8_any_t __attribute__((ext_vector_type(8), aligned(2)));  // half8_t at any half's address

template <class E, class = void>
struct Activates : std::false_type {};
template <class E>
struct Activates<E, std::void_t<decltype(&E::activate)>> : std::true_type {};

// One row sub-tile (32 rows) per pass: a wavefront stages TN * 4 KB.
template <int TME, int TN>
struct RowwiseEpilogueCfg {
  static constexpr int RT = 1;
  static constexpr int kPitch = TN * 128;                 // bytes per staged row (fp32)
  static constexpr int kBytesPerWave = RT * 32 * kPitch;
};

// acc[i][t]: sub-tile (i, t) of a wavefront's TME x TN sub-tiles whose first element is
// (m_base, n_base).  `stage`: this wavefront's kBytesPerWave bytes of LDS that nobody else
// touches.
template <class Epilogue, int TME, int TN>
__device__ __forceinline__ void store_tile_rowwise(const float16_t (&acc)[TME][TN], const Epilogue& epilogue,
                                                   half_t* __restrict__ Y, int M, int N, int m_base,
                                                   int n_base, unsigned char* stage, int lane) {
  using Cfg = RowwiseEpilogueCfg<TME, TN>;
  constexpr int RT = Cfg::RT, kPitch = Cfg::kPitch;
  const int lj = lane & 31, lh = lane >> 5;
  // activation pass: a lane stays on one column
  constexpr int kRowsPerPass = 64 / (TN * 32);
  const int act_col = lane % (TN * 32), act_n = min(n_base + act_col, N - 1);
  float col_bias = 0.0f;
  if constexpr (Activates<Epilogue>::value) {
    static_assert(TN <= 2, "a wavefront covers at least one row per pass");
    if (epilogue.activates()) col_bias = epilogue.column_bias(act_n);
  }
#pragma unroll
  for (int i0 = 0; i0 < TME; i0 += RT) {
#pragma unroll
    for (int ii = 0; ii < RT; ++ii) {
      if (i0 + ii < TME) {
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = ii * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
            *reinterpret_cast<float*>(stage + row * kPitch + (t * 32 + lj) * 4) = acc[i0 + ii < TME ? i0 + ii : 0][t][r];
          }
      }
    }
    // LDS operations of one wavefront execute in order: no barrier between write and read
    if constexpr (Activates<Epilogue>::value) {
      if (epilogue.activates()) {
#pragma unroll 4
        for (int it = 0; it < 16 * TN; ++it) {
          const int row = it * kRowsPerPass + lane / (TN * 32);
          float* const v = reinterpret_cast<float*>(stage + row * kPitch + act_col * 4);
          *v = epilogue.activate(*v, col_bias, min(m_base + i0 * 32 + row, M - 1), act_n);
        }
      }
    }
    constexpr int kGroupsPerRow = TN * 4;  // groups of 8 columns
    constexpr int kIters = RT * 32 * kGroupsPerRow / 64;
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      const int c = it * 64 + lane;
      const int row = c / kGroupsPerRow, cc = c % kGroupsPerRow;
      const float4_t v0 = *reinterpret_cast<const float4_t*>(stage + row * kPitch + cc * 32);
      const float4_t v1 = *reinterpret_cast<const float4_t*>(stage + row * kPitch + cc * 32 + 16);
      const int m = m_base + i0 * 32 + row;
      const int n = n_base + cc * 8;
      if (row < (TME - i0) * 32 && m < M && n < N) {
        const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        half_t* const y = Y + (int64_t)m * N + n;
        if (n + 8 <= N) {
          *reinterpret_cast<half8_any_t*>(y) = epilogue.apply8(v, m, n);
        } else if constexpr (!Activates<Epilogue>::value) {
          const float* const staged = reinterpret_cast<const float*>(stage + row * kPitch + cc * 32);
#pragma unroll 1
          for (int e = 0; e < N - n; ++e) y[e] = epilogue(staged[e], m, n + e);
        }
      }
    }
  }
}

}  // namespace wq
#endif  // RELAX_AMD_CSRC_GEMM_EPILOGUE_H_
