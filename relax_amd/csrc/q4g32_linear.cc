// Shape-based choice between the decode GEMV, the small-batch kernel and the MFMA GEMM for format A.
#include <cstdint>

#include "q4g32_dispatch.h"
#include "wq_host.h"

extern "C" int wq_q4g32_linear(const uint32_t* W, const uint16_t* S, const uint16_t* x,
                               const uint16_t* bias, const uint16_t* residual, uint16_t* y,
                               int64_t M, int64_t N, int64_t K, wq_stream_t stream) {
  // one or two rows: the VALU streaming kernel; up to 64 rows: still one pass over the
  // weights, products on the matrix cores; beyond that the tiled GEMM.  A kernel whose
  // preconditions the operands do not meet (K range, scale alignment) is passed over
  // for the next one that serves the call.
  const bool gemv_ok = K <= 32768;
  // K % 64 == 32 has a form of the small-batch kernel with its own scale addressing; before it, 3 .. 8 rows went
  // through the streaming kernel in pairs and more through the GEMM (N = 11008, K = 4064: M = 3 14.6 -> 10.7 us,
  // M = 8 29.4 -> 10.7, M = 19 65 -> 19, M = 64 66 -> 25); like the kernel they left, up to 8 rows take the weights
  // unrounded
  const bool half_step = K > 0 && K % 64 == 32 && wq::q4g32_half_step_rows_ok(x, N);
  const bool small_ok = (K % 64 == 0 || half_step) && (reinterpret_cast<uintptr_t>(S) & 3u) == 0;
  const auto small_batch = [&](const uint16_t* x_, const uint16_t* residual_, uint16_t* y_, int64_t M_) {
    if (half_step) return wq::q4g32_half_step_rows(W, S, x_, bias, residual_, y_, M_, N, K, (hipStream_t)stream);
    return wq_q4g32_small_batch(W, S, x_, bias, residual_, y_, M_, N, K, stream);
  };
  // (two rows of more than 8192 columns: the streaming kernel's two-row form is the slower one there; N = 4096,
  // K = 11008: 15.5 against 10.9 us, N = 8192, K = 28672: 56 against 37 us)
  const bool two_long_rows = M == 2 && K > 8192 && small_ok;
  if (M <= 2 && gemv_ok && !two_long_rows) return wq_q4g32_gemv(W, S, x, bias, residual, y, M, N, K, stream);
  if (M <= WQ_SMALL_BATCH_MAX_M && small_ok) return small_batch(x, residual, y, M);
  // up to 128 rows of a small matrix: the tiled GEMM would have too few tiles for 256
  // CUs; two passes of the small-batch kernel are faster
  if (M > WQ_SMALL_BATCH_MAX_M && M <= 2 * WQ_SMALL_BATCH_MAX_M && small_ok && N <= 8192) {
    const int64_t m0 = WQ_SMALL_BATCH_MAX_M;
    if (int rc = small_batch(x, residual, y, m0)) return rc;
    return small_batch(x + m0 * K, residual ? residual + m0 * N : nullptr, y + m0 * N, M - m0);
  }
  if (M <= WQ_GEMV_MAX_M && gemv_ok) return wq_q4g32_gemv(W, S, x, bias, residual, y, M, N, K, stream);
  return wq_q4g32_gemm(W, S, x, bias, residual, y, M, N, K, stream);
}
