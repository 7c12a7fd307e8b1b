// Format A (q4f16_1) small-batch entry: the shared small-batch kernel with the
// group-32 int4 weight policy.
#include "held_gemm.h"
#include "q4g32_common.h"
#include "q4g32_dispatch.h"
#include "skinny_gemm.h"

namespace wq {

// W uint32 [N, K/8], S fp16 [N, K/32]: the 32 codes at k0 are the 16 bytes at
// row + k0/2; their scale is S[n][k0/32], fetched as the aligned pair that holds it.
struct Q4G32SkinnyPolicy {
  static constexpr int kPieces = 1;
  static constexpr bool kScaleDma = true;
  static constexpr bool kCanScaleBlock = true;
  static constexpr bool kXreg = false;  // (K % 64 == 0: held_gemm.h)
  struct Args {
    const uint32_t* W;
    const half_t* S;
  };
  struct Lane {
    const char* w;
    const char* s;
  };
  __device__ __forceinline__ static void init(Lane& l, const Args& a, int n, int K, int) {
    l.w = reinterpret_cast<const char*>(a.W + (int64_t)n * (K >> 3));
    l.s = reinterpret_cast<const char*>(a.S + (int64_t)n * (K >> 5));
  }
  __device__ __forceinline__ static const char* w_addr(const Lane& l, int k0, int) { return l.w + (k0 >> 1); }
  __device__ __forceinline__ static const char* s_addr(const Lane& l, int k0) { return l.s + ((k0 >> 5) & ~1) * 2; }
  __device__ __forceinline__ static const char* s_pair_addr(const Lane& l, int k0) { return s_addr(l, k0); }
  static constexpr int kStepStride = 64;
  __device__ __forceinline__ static const char* s_lane(const Lane& l) { return l.s; }
  __device__ __forceinline__ static uint32_t s_rel(const Lane&, int k0) { return ((k0 >> 5) & ~1) * 2; }
  static int64_t s_reach(const Args&, int64_t, int64_t K) { return K; }
  // rows of K/16 bytes: every 8 scales are 16 aligned bytes when K % 256 == 0 and S is aligned
  static bool scale_block_ok(const Args& a, int64_t K) {
    return K % 256 == 0 && (reinterpret_cast<uintptr_t>(a.S) & 15u) == 0;
  }
  static bool pair_aligned(const Args& a) { return (reinterpret_cast<uintptr_t>(a.S) & 3u) == 0; }
  __device__ __forceinline__ static half_t pick_scale(const Lane&, half2_t pair, int kq) { return (kq & 1) ? pair.y : pair.x; }
  using Scale = half_t;
  __device__ __forceinline__ static half_t const_scale(const Lane&) { return (half_t)0.0f; }
  __device__ __forceinline__ static half_t null_scale() { return (half_t)0.0f; }
  __device__ __forceinline__ static void dequant(const uint4_t* pieces, half_t s, half8_t out[4]) {
    const half2_t s2 = {s, s};
    const uint32_t words[4] = {pieces[0].x, pieces[0].y, pieces[0].z, pieces[0].w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      half2_t d[4];
      q4_word_dequant_natural(words[t], s2, d);
      out[t] = half8_t{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
    }
  }
};

// The same for K % 64 == 32 and an even N: a row of S holds an odd number of scales, so which half of the
// aligned pair a scale is depends on the row as well.  (An odd N would have the pair of its very last scale end
// past S.)
struct Q4G32OddGroupsSkinnyPolicy : Q4G32SkinnyPolicy {
  static constexpr bool kCanScaleBlock = false;
  static constexpr bool kOddStart = true;
  static constexpr bool kXreg = true;
  struct Lane : Q4G32SkinnyPolicy::Lane {
    int odd;  // parity of the row
  };
  __device__ __forceinline__ static void init(Lane& l, const Args& a, int n, int K, int N) {
    Q4G32SkinnyPolicy::init(l, a, n, K, N);
    l.odd = n & 1;
  }
  __device__ __forceinline__ static uint32_t s_rel(const Lane& l, int k0) { return ((k0 >> 5) - (((k0 >> 5) + l.odd) & 1)) * 2; }
  __device__ __forceinline__ static const char* s_addr(const Lane& l, int k0) { return l.s + (int)s_rel(l, k0); }
  __device__ __forceinline__ static const char* s_pair_addr(const Lane& l, int k0) { return s_addr(l, k0); }
  // the lane's group is 4 * step + kq
  __device__ __forceinline__ static half_t pick_scale(const Lane& l, half2_t pair, int kq) {
    return ((kq + l.odd) & 1) ? pair.y : pair.x;
  }
};

// Up to 8 rows of such a K: (code - 7) * scale is not rounded to fp16, as in the streaming kernel that serves them
// elsewhere (against 64 bits, K = 4064: 2.06e-4, most of it the rounding of y; with rounded weights 2.75e-4).
// M = 8, streaming kernel / this / rounded weights: N = 11008, K = 4064 29.4 / 10.6 / 10.4 us, N = 4096, K = 11040
// 45.3 / 11.8 / 11.1 us, N = 28672, K = 8160 112 / 44.2 / 43.1 us.
struct Q4G32OddGroupsExactSkinnyPolicy : Q4G32OddGroupsSkinnyPolicy {
  __device__ __forceinline__ static half8_t codes8(uint32_t word) {
    const half2_t one = {(half_t)1.0f, (half_t)1.0f};
    half2_t d[4];
    q4_word_dequant_natural(word, one, d);
    return half8_t{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
  }
};

int q4g32_half_step_rows(const uint32_t* W, const uint16_t* S, const uint16_t* x, const uint16_t* bias,
                         const uint16_t* residual, uint16_t* y, int64_t M, int64_t N, int64_t K,
                         hipStream_t stream) {
  if (M == 0) return WQ_OK;
  WQ_REQUIRE(M > 0 && M <= WQ_SMALL_BATCH_MAX_M && K > 0 && K % 64 == 32 && q4g32_half_step_rows_ok(x, N),
             "wq_q4g32_linear: M=%lld, N=%lld, K=%lld", (long long)M, (long long)N, (long long)K);
  WQ_REQUIRE(W && S && x && y, "wq_q4g32_linear: null pointer");
  WQ_REQUIRE(aligned16(W) && (reinterpret_cast<uintptr_t>(S) & 3u) == 0,
             "wq_q4g32_linear: W must be 16-byte aligned, S 4-byte aligned");
  WQ_REQUIRE(N < (1ll << 30) && K < (1ll << 30), "wq_q4g32_linear: too large");
  const Q4G32OddGroupsSkinnyPolicy::Args pargs{W, (const half_t*)S};
  const Q4G32Epilogue epi{(const half_t*)bias, (const half_t*)residual, (int)N};
  if (M <= 8)
    return launch_skinny_auto<Q4G32OddGroupsExactSkinnyPolicy, Q4G32Epilogue>("wq_q4g32_linear", pargs, x, y, epi, M,
                                                                              N, K, stream);
  return launch_skinny_auto<Q4G32OddGroupsSkinnyPolicy, Q4G32Epilogue>("wq_q4g32_linear", pargs, x, y, epi, M, N,
                                                                       K, stream);
}

}  // namespace wq

// Small-batch entry: 1 <= M <= 64, K % 64 == 0.  Called by wq_q4g32_linear.
extern "C" int wq_q4g32_small_batch(const uint32_t* W, const uint16_t* S, const uint16_t* x,
                                    const uint16_t* bias, const uint16_t* residual, uint16_t* y,
                                    int64_t M, int64_t N, int64_t K, wq_stream_t stream_) {
  using namespace wq;
  hipStream_t stream = (hipStream_t)stream_;
  WQ_REQUIRE(M >= 0 && N >= 0 && K >= 0, "wq_q4g32_small_batch: negative dimension");
  WQ_REQUIRE(M <= WQ_SMALL_BATCH_MAX_M, "wq_q4g32_small_batch: M=%lld > %d", (long long)M,
             WQ_SMALL_BATCH_MAX_M);
  WQ_REQUIRE(K % 64 == 0, "wq_q4g32_small_batch: K=%lld must be a multiple of 64", (long long)K);
  if (M == 0 || N == 0) return WQ_OK;
  WQ_REQUIRE(K > 0, "wq_q4g32_small_batch: K must be positive");
  WQ_REQUIRE(W && S && x && y, "wq_q4g32_small_batch: null pointer");
  WQ_REQUIRE(aligned16(W) && aligned16(x) && (reinterpret_cast<uintptr_t>(S) & 3u) == 0,
             "wq_q4g32_small_batch: W and x must be 16-byte aligned, S 4-byte aligned");
  WQ_REQUIRE(N < (1ll << 30) && K < (1ll << 30), "wq_q4g32_small_batch: too large");
  const Q4G32Epilogue epi{(const half_t*)bias, (const half_t*)residual, (int)N};
  if (held_takes(kHeldQ4, M, N, K))
    return launch_held<kHeldQ4, Q4G32Epilogue>("wq_q4g32_small_batch", HeldArgs{(const char*)W, (const char*)S, 0, 1}, x, y,
                                               epi, M, N, K, stream);
  const Q4G32SkinnyPolicy::Args pargs{W, (const half_t*)S};
  return launch_skinny_auto<Q4G32SkinnyPolicy, Q4G32Epilogue>("wq_q4g32_small_batch", pargs, x, y, epi,
                                                             M, N, K, stream);
}
