// The LDS-staged GEMM's weight policies of formats A and B, and its 256 x 256 tiles (configuration 11) where they are
// compiled by themselves (gemm_256.hip).
#ifndef RELAX_AMD_CSRC_GEMM_256_H_
#define RELAX_AMD_CSRC_GEMM_256_H_

#include "intb_common.h"
#include "mfma_gemm_lds.h"
#include "q4g32_common.h"

namespace wq {

// Weight policy of the fully LDS-staged kernel (mfma_gemm_lds.h) for format A: per K-step a
// column is 32 bytes of codes (chunk (n, h) of the B tile = 16 bytes = one scale group) and two
// scales (4 bytes, staged in LDS with the codes).
struct Q4G32LdsPolicy {
  static constexpr bool kFineTail = true;  // a last round of few tiles may be cut into eight row slices
  static constexpr int kColBytes = 32;
  static constexpr int kScaleBytes = 4;
  static constexpr int kStepStride = 32;
  struct Args {
    const uint32_t* W;
    const half_t* S;
  };
  struct Frag {
    uint4_t w;
  };
  using Scale = half_t;  // the group's scale
  __device__ __forceinline__ static const char* b_src(const Args& a, int n0, int q, int N, int K) {
    const int n = q >> 1, h = q & 1;
    return reinterpret_cast<const char*>(a.W + (int64_t)min(n0 + n, N - 1) * (K >> 3)) + h * 16;
  }
  __device__ __forceinline__ static const char* s_src(const Args& a, int n, int K) {
    return reinterpret_cast<const char*>(a.S + (int64_t)n * (K >> 5));
  }
  __device__ __forceinline__ static int64_t s_offset(const Args&, int ks) { return (int64_t)ks * 4; }
  __device__ __forceinline__ static Scale read_scale(const unsigned char* p, int lh) {
    return *reinterpret_cast<const half_t*>(p + lh * 2);
  }
  __device__ __forceinline__ static Scale const_scale(const Args&, int) { return (half_t)0.0f; }
  __device__ __forceinline__ static void read(Frag& f, const unsigned char* bslot, int n_local, int lh) {
    f.w = *reinterpret_cast<const uint4_t*>(bslot + (n_local * 2 + lh) * 16);
  }
  __device__ __forceinline__ static uint32_t pair_bits(const Frag& f, int kk, int j) {
    const uint32_t word = kk == 0 ? f.w.x : kk == 1 ? f.w.y : kk == 2 ? f.w.z : f.w.w;
    const half2_t off = {(half_t)1031.0f, (half_t)1031.0f};
    return as_u32(as_half2(q4_pair_bits_natural(word, j)) - off);
  }
  __device__ __forceinline__ static half2_t pair_finish(uint32_t bits, Scale s) { return as_half2(bits) * half2_t{s, s}; }
  __device__ __forceinline__ static half2_t pair(const Frag& f, int kk, int j, Scale s) { return pair_finish(pair_bits(f, kk, j), s); }
};

// The same with the weights in registers, from K = 256 on (the scales of four steps are fetched at a time).
struct Q4G32RegPolicy : Q4G32LdsPolicy {
  static constexpr bool kRegB = true, kFourScales = true;
  __device__ __forceinline__ static const char* b_base(const Args& a, int n0, int K) {
    return reinterpret_cast<const char*>(a.W + (int64_t)n0 * (K >> 3));
  }
  __device__ __forceinline__ static uint32_t b_lane(int n, int n0, int lh, int K) { return (uint32_t)(n - n0) * (uint32_t)(K >> 1) + lh * 16; }
  __device__ __forceinline__ static const char* s_base(const Args& a, int n0, int K) { return s_src(a, n0, K); }
  __device__ __forceinline__ static uint32_t s_lane(const Args&, int n, int n0, int K) { return (uint32_t)(n - n0) * (uint32_t)(K >> 4); }
};

// Weight policy of the fully LDS-staged kernel (mfma_gemm_lds.h) for the preprocessed layouts
// with per-column scales.  A K-step (one 64-row tile) of I = 2 (int8) or 4 (int4) interleaved
// columns is 128 contiguous bytes, so the B tile is fetched in whole 128-byte lines; the scale
// of a column never changes, stays in a register and is applied to the sums: on the weights it was a third of the instructions
// that unpack them, and a rounding each (N = 11008, K = 4096, M = 2048 int8 / int4 184.6 / 185.0 -> 172.3 / 167.4 us; N = 28672,
// K = 8192, M = 128 83.6 / 74.1 -> 82.3 / 69.8, where a CU has one tile and waits for its loads; error against 64 bits
// 2.94e-4 / 2.76e-4 -> 2.07e-4).
// GROUPED (scales fp16 [K/64, N], one per column and K-step): a lane stages the 4 bytes that hold
// the scales of its column and the neighbouring one, and the reader takes its half.
template <int NBIT, bool GROUPED = false>
struct IntbLdsPolicy {
  static constexpr int I = NBIT == 8 ? 2 : 4;
  static constexpr int kColBytes = 128 / I;
  static constexpr int kScaleBytes = GROUPED ? 4 : 0;
  static constexpr bool kColumnScale = !GROUPED;  // to the sums, in fp32: the weights are the codes, exact
  static constexpr int kStepStride = 128;
  struct Args {
    const uint4_t* B;
    const half_t* scales;
    int N;
  };
  struct Frag {
    uint4_t w[NBIT == 8 ? 2 : 1];
  };
  __device__ __forceinline__ static const char* b_src(const Args& a, int n0, int q, int N, int K) {
    const int group = min(n0 / I + (q >> 3), N / I - 1);  // columns past N re-read the last group
    return reinterpret_cast<const char*>(a.B) + ((int64_t)group * (K >> 6)) * 128 + (q & 7) * 16;
  }
  using Scale = half_t;  // the column's scale
  __device__ __forceinline__ static const char* s_src(const Args& a, int n, int) {
    return reinterpret_cast<const char*>(a.scales + (n & ~1));  // the aligned pair of columns (N is even)
  }
  __device__ __forceinline__ static int64_t s_offset(const Args& a, int ks) { return (int64_t)ks * a.N * 2; }
  // p = the 4 staged bytes of the lane's column; columns are staged 4 bytes apart from an 8-byte
  // aligned base, so bit 2 of the address is the parity of the column
  __device__ __forceinline__ static Scale read_scale(const unsigned char* p, int) {
    return *reinterpret_cast<const half_t*>(p + ((reinterpret_cast<uintptr_t>(p) & 4) >> 1));
  }
  __device__ __forceinline__ static Scale const_scale(const Args& a, int n) {
    return a.scales[n];
  }
  __device__ __forceinline__ static void read(Frag& f, const unsigned char* bslot, int n_local, int lh) {
    if (NBIT == 8) {
      const unsigned char* p = bslot + ((n_local >> 1) * 8 + (n_local & 1) * 4 + 2 * lh) * 16;
      f.w[0] = *reinterpret_cast<const uint4_t*>(p);
      f.w[NBIT == 8 ? 1 : 0] = *reinterpret_cast<const uint4_t*>(p + 16);
    } else {
      f.w[0] = *reinterpret_cast<const uint4_t*>(bslot + ((n_local >> 2) * 8 + (n_local & 3) * 2 + lh) * 16);
    }
  }
  // int8: piece kk/2 holds 16 k; word j of it holds k = 2j, 2j+1 (bytes 0, 2) and 2j+8, 2j+9 (bytes 1, 3).
  // int4: word j holds k = 2j + 8i, 2j + 8i + 1 in nibbles i, i + 4.
  __device__ __forceinline__ static uint32_t pair_bits(const Frag& f, int kk, int j) {
    if (NBIT == 8) {
      const uint4_t& p = f.w[NBIT == 8 ? (kk >> 1) : 0];
      const uint32_t word = j == 0 ? p.x : j == 1 ? p.y : j == 2 ? p.z : p.w;
      return minus(__builtin_amdgcn_perm(0x64646464u, word, (kk & 1) ? 0x04030401u : 0x04020400u), 1152.0f);  // 1024 + u8
    }
    const uint32_t word = j == 0 ? f.w[0].x : j == 1 ? f.w[0].y : j == 2 ? f.w[0].z : f.w[0].w;
    return minus(and_or_b(word >> (4 * kk), 0x000F000Fu, 0x64006400u), 1032.0f);                                // 1024 + u4
  }
  __device__ __forceinline__ static uint32_t minus(uint32_t bits, float o) { return as_u32(as_half2(bits) - half2_t{(half_t)o, (half_t)o}); }
  __device__ __forceinline__ static half2_t pair_finish(uint32_t bits, Scale s) {
    return kColumnScale ? as_half2(bits) : as_half2(bits) * half2_t{s, s};
  }
  __device__ __forceinline__ static half2_t pair(const Frag& f, int kk, int j, Scale s2) { return pair_finish(pair_bits(f, kk, j), s2); }
};

int q4g32_gemm_256(const char* who, const Q4G32RegPolicy::Args& wargs, const uint16_t* x, uint16_t* y,
                   const Q4G32Epilogue& ep, int64_t M, int64_t N, int64_t K, hipStream_t stream);

template <int NBIT, bool GROUPED>  // defined for int4, and for int8 with a scale per 64
int intb_gemm_256(const char* who, const typename IntbLdsPolicy<NBIT, GROUPED>::Args& wargs, const uint16_t* A,
                  uint16_t* C, const IntbGemmEpilogue& ep, int64_t m, int64_t n, int64_t k, hipStream_t stream);

}  // namespace wq
#endif  // RELAX_AMD_CSRC_GEMM_256_H_
