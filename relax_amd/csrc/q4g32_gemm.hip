// Format A prefill GEMM: y[m,n] = sum_k x[m,k] * ((code[n,k] - 7) * S[n,k/32]).
// The kernel is the shared MFMA GEMM (mfma_gemm.h); this file supplies the weight
// loader for the q4f16_1 layout and the epilogue of the reference's prefill
// PrimFunc (tests/python/dlight/test_gpu_matmul.py:378-401).
#include "mfma_gemm.h"
#include "gemm_256.h"
#include "q4g32_common.h"

namespace wq {

// Lane (j, h) of a K-step needs k = 32h..32h+31 of weight row n: exactly one scale
// group, i.e. 4 consecutive words (16 bytes) of W and one scale; word kk is the
// B operand of MFMA kk.
struct Q4G32Loader {
  static constexpr bool kPairA = true;  // q4_word_dequant yields the (i, i+4) pairing
  struct Args {
    const uint32_t* W;
    const half_t* S;
  };
  struct Lane {
    const uint4_t* w;
    const half_t* s;
  };
  struct Frag {
    uint4_t w;
    half_t s;
  };
  __device__ __forceinline__ static void init(Lane& l, const Args& a, int n, int lh, int K, int) {
    l.w = reinterpret_cast<const uint4_t*>(a.W + (int64_t)n * (K >> 3)) + lh;
    l.s = a.S + (int64_t)n * (K >> 5) + lh;
  }
  __device__ __forceinline__ static void load(Frag& f, const Lane& l, const Args&, int ks, int lh, int K,
                              bool ktail) {
    if (ktail && (ks * 2 + lh) >= (K >> 5)) {  // the last step may hold a single group
      f.w = uint4_t{0x77777777u, 0x77777777u, 0x77777777u, 0x77777777u};  // code 7 -> weight 0
      f.s = (half_t)0.0f;
    } else {
      f.w = l.w[ks * 2];
      f.s = l.s[ks * 2];
    }
  }
  __device__ __forceinline__ static void dequant(const Frag& f, half8_t out[4]) {
    const half2_t s2 = {f.s, f.s};
    const uint32_t ws[4] = {f.w.x, f.w.y, f.w.z, f.w.w};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      half2_t d[4];
      q4_word_dequant(ws[kk], s2, d);
      out[kk] = half8_t{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
    }
  }
};

// Q4G32LdsPolicy for K % 64 == 32.  A row of S then holds an odd number G of scales: in odd rows the pair of a K-step
// straddles two aligned words, so both are staged (in even rows the first one twice), and the last 32 k are half
// a step.  Nothing past a row is read: the steps end one scale before its end, so the second word of an odd row
// ends with that row's last scale, at the latest.
// Before, such a K took the register-staged kernel, which cannot overlap its loads as deeply: M = 2048,
// N = 11008, K = 4064: 374 -> 201 us; M = 200: 91 -> 43 us.
struct Q4G32HalfStepPolicy : Q4G32LdsPolicy {
  static constexpr bool kFineTail = false;
  static constexpr int kScaleBytes = 8;
  __device__ __forceinline__ static const char* s_src(const Args& a, int n, int K) {
    return reinterpret_cast<const char*>(a.S + (((int64_t)n * (K >> 5)) & ~(int64_t)1));
  }
  __device__ __forceinline__ static const char* s_src2(const Args& a, int n, int K) {
    return s_src(a, n, K) + ((n & 1) ? 4 : 0);
  }
  // n_local has the parity of the column: tiles start at multiples of 128
  __device__ __forceinline__ static Scale read_scale2(const unsigned char* p, int plane, int n_local, int lh) {
    return *reinterpret_cast<const half_t*>(p + ((n_local & 1) ? (lh ? plane : 2) : 2 * lh));
  }
  __device__ __forceinline__ static void half_step(const Args& a, int n, int k0, int K, int lh, half8_t out[2]) {
    const uint32_t* const w = a.W + (int64_t)n * (K >> 3) + (k0 >> 3) + lh;
    const half_t s = a.S[(int64_t)n * (K >> 5) + (k0 >> 5)];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const uint32_t word = w[2 * c];
      half2_t d[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = half2_t{s, s} * (as_half2(q4_pair_bits_natural(word, j)) - half2_t{(half_t)1031.0f, (half_t)1031.0f});
      out[c] = half8_t{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
    }
  }
};

}  // namespace wq

// Tile shape override for measurement (0 = choose from the problem shape).
int wq_gemm_cfg_override() { return wq::tuning().gemm_cfg; }

extern "C" int wq_q4g32_gemm(const uint32_t* W, const uint16_t* S, const uint16_t* x,
                             const uint16_t* bias, const uint16_t* residual, uint16_t* y, int64_t M,
                             int64_t N, int64_t K, wq_stream_t stream_) {
  using namespace wq;
  hipStream_t stream = (hipStream_t)stream_;
  WQ_REQUIRE(M >= 0 && N >= 0 && K >= 0, "wq_q4g32_gemm: negative dimension");
  WQ_REQUIRE(K % 32 == 0, "wq_q4g32_gemm: K=%lld must be a multiple of the group size 32",
             (long long)K);
  if (M == 0 || N == 0) return WQ_OK;
  WQ_REQUIRE(K > 0, "wq_q4g32_gemm: K must be positive");
  WQ_REQUIRE(W && S && x && y, "wq_q4g32_gemm: null pointer");
  WQ_REQUIRE(aligned16(W) && aligned16(x), "wq_q4g32_gemm: W and x must be 16-byte aligned");
  WQ_REQUIRE(M < (1ll << 30) && N < (1ll << 30) && K < (1ll << 30), "wq_q4g32_gemm: too large");
  int cfg = tuning().gemm_cfg                       ? tuning().gemm_cfg
            : q4_lds_k_halves(M, N, K, cu_count()) ? 19
                                                   : choose_q4_lds_cfg(M, N, cu_count());
  const Q4G32Loader::Args bargs{W, (const half_t*)S};
  const Q4G32LdsPolicy::Args largs{W, (const half_t*)S};
  const Q4G32Epilogue ep{(const half_t*)bias, (const half_t*)residual, (int)N};
  // 11..19: the fully LDS-staged kernel (needs 4-byte aligned S and 32-bit offsets inside a tile); K % 64 == 32 has the three shapes that the
  // choice above takes for most problems
  const bool lds_ok = ((uintptr_t)S & 3u) == 0 && K < kLdsGemmMaxK;
  if (cfg >= 11 && K % 64 == 32 && lds_ok) {
    switch (cfg) {
      case 17: case 19: return launch_gemm_lds<Q4G32HalfStepPolicy, Q4G32Epilogue, 4, 1, 1, 4, 2>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 12: case 13:
      case 18: return launch_gemm_lds<Q4G32HalfStepPolicy, Q4G32Epilogue, 8, 1, 1, 4, 1>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 11: case 14: return launch_gemm_lds<Q4G32HalfStepPolicy, Q4G32Epilogue, 8, 2, 1, 4, 1>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      default: return fail(WQ_EINVAL, "wq_q4g32_gemm: unknown tile configuration %d", cfg);
    }
  }
  if (cfg >= 11 && K % 64 == 0 && lds_ok) {
    if (cfg == 15 || cfg == 16 || cfg > 19) return fail(WQ_EINVAL, "wq_q4g32_gemm: unknown tile configuration %d", cfg);
    // fewer steps than the weights are requested ahead; 256 x 256 tiles up to K = 320, where filling that pipeline, with
    // one workgroup per CU, costs more than it brings (N = 22016: K = 256, M = 2048 51.2 -> 42.6 us, M = 8192 174.7 -> 160.0,
    // K = 320, M = 1024 31.9 -> 29.9; 7 % on average over N = 4096 .. 28672, M = 512 .. 8192, N = 16384, K = 256,
    // M = 4096 5 % slower; at K = 384 as many shapes lose as gain)
    if (K < 256 || (K <= 320 && cfg == 11 && !tuning().gemm_cfg))
      return launch_gemm_lds<Q4G32LdsPolicy, Q4G32Epilogue, 4, 1, 1, 4, 2>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
    if (cfg == 19 && K % 128 != 0) cfg = 17;
    using P = Q4G32RegPolicy;
    switch (cfg) {
      case 11: return q4g32_gemm_256("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 12: return launch_gemm_lds<P, Q4G32Epilogue, 4, 2, 1, 4, 2>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 13: return launch_gemm_lds<P, Q4G32Epilogue, 4, 2, 2, 2, 2>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 14: return launch_gemm_lds<P, Q4G32Epilogue, 4, 4, 2, 2, 1>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 17: return launch_gemm_lds<P, Q4G32Epilogue, 4, 1, 1, 4, 2>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      case 18: return launch_gemm_lds<P, Q4G32Epilogue, 8, 1, 1, 4, 1>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
      default: return launch_gemm_lds<P, Q4G32Epilogue, 4, 1, 1, 4, 2, 2>("wq_q4g32_gemm", largs, x, y, ep, M, N, K, stream);
    }
  }
  if (cfg >= 11) cfg = (cfg == 17 || cfg == 19) ? 4 : (cfg == 11 || cfg == 14) ? 1 : 2;  // 12, 13, 18 -> 128 x 256  // not eligible: register-staged kernel, same tile
  return launch_mfma_gemm_cfg<Q4G32Loader, Q4G32Epilogue>(cfg, "wq_q4g32_gemm", bargs, x, y, ep, M,
                                                          N, K, stream);
}
