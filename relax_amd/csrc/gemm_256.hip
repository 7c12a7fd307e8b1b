// 256 x 256 tiles of the LDS-staged GEMM (mfma_gemm_lds.h), one wavefront per SIMD.  In a file of their own because the
// build aligns its loops: the main loop is the same code wherever it lies, but from the middle of an instruction cache line
// it takes 1 % longer (q4f16_1, N = 22016, K = 4096, M = 8192: 1302 us, aligned 1287; fpA_intB int4 with a scale per 64,
// N = 28672, K = 8192, M = 2048: 870 -> 862).  Others lose by it and stay where they are: int8 per column (N = 28672,
// K = 8192, M = 2048: 830 -> 848 us) and the smaller tiles (q4f16_1, N = K = 5120, M = 640, 256 x 128: 48.9 -> 49.6 us).
#include "gemm_256.h"

namespace wq {

int q4g32_gemm_256(const char* who, const Q4G32RegPolicy::Args& wargs, const uint16_t* x, uint16_t* y,
                   const Q4G32Epilogue& ep, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  return launch_gemm_lds<Q4G32RegPolicy, Q4G32Epilogue, 8, 2, 1, 4, 1>(who, wargs, x, y, ep, M, N, K, stream);
}

template <int NBIT, bool GROUPED>
int intb_gemm_256(const char* who, const typename IntbLdsPolicy<NBIT, GROUPED>::Args& wargs, const uint16_t* A,
                  uint16_t* C, const IntbGemmEpilogue& ep, int64_t m, int64_t n, int64_t k, hipStream_t stream) {
  return launch_gemm_lds<IntbLdsPolicy<NBIT, GROUPED>, IntbGemmEpilogue, 8, 2, 1, 4, 1>(who, wargs, A, C, ep, m, n, k,
                                                                                        stream);
}

#define WQ_INTB_256(NBIT, GROUPED)                                                                                  \
  template int intb_gemm_256<NBIT, GROUPED>(const char*, const IntbLdsPolicy<NBIT, GROUPED>::Args&, const uint16_t*, \
                                            uint16_t*, const IntbGemmEpilogue&, int64_t, int64_t, int64_t, hipStream_t);
WQ_INTB_256(8, true)
WQ_INTB_256(4, false)
WQ_INTB_256(4, true)
#undef WQ_INTB_256

}  // namespace wq
