// Declarations shared by the format-B GEMV and GEMM translation units.
#ifndef RELAX_AMD_CSRC_INTB_COMMON_H_
#define RELAX_AMD_CSRC_INTB_COMMON_H_

#include "gemm_epilogue.h"
#include "wq_device.h"
#include "wq_host.h"

namespace wq {

// Fused epilogue of the mixed-input GEMM: act(acc + bias) [binary residual] [unary].
// bias_stride == 0 broadcasts bias[n] over rows.  activation / binary_op / unary_op
// are the WQ_ACT_* / WQ_BIN_* / WQ_UN_* selectors.
struct IntbEpilogue {
  const half_t* bias;
  const half_t* residual;
  int64_t bias_stride;
  int activation, binary_op, unary_op;
};

// Streaming kernel for m <= 4 (intb_gemv.hip).  `group` is 0 (per column) or 64.
int intb_gemv_dispatch(const uint16_t* A, const int8_t* B, const uint16_t* scales, uint16_t* C,
                       int64_t m, int64_t n, int64_t k, int64_t group, int nbit,
                       const IntbEpilogue& ep, hipStream_t stream);

// Wavefronts that kernel's launch for one or two rows would have: it gives a wavefront whole columns, so a
// narrow matrix leaves the machine short of them.
int64_t intb_gemv_wavefronts(int64_t m, int64_t n, int64_t group, int nbit);

// Matrix-core streaming kernel for 1 <= m <= 64 (intb_skinny.hip).
int intb_small_batch_dispatch(const uint16_t* A, const int8_t* B, const uint16_t* scales, uint16_t* C,
                              int64_t m, int64_t n, int64_t k, int64_t group, int nbit,
                              const IntbEpilogue& ep, hipStream_t stream);

#ifdef __HIPCC__
// act(acc + bias) [binary residual] [unary], all in fp32, one rounding at the store
struct IntbGemmEpilogue {
  IntbEpilogue e;
  int N;
  // silu and gelu: bias and activation in a pass of their own (gemm_epilogue.h), relu with the store
  __device__ bool activates() const { return e.activation >= 2; }
  __device__ float column_bias(int n) const { return e.bias && !e.bias_stride ? (float)e.bias[n] : 0.0f; }
  __device__ float activate(float v, float column_bias, int m, int n) const {
    if (e.bias) v += e.bias_stride ? (float)e.bias[(int64_t)m * e.bias_stride + n] : column_bias;
    return apply_activation(v, e.activation);
  }
  __device__ half_t operator()(float v, int m, int n) const {
    v = activate(v, column_bias(n), m, n);
    if (e.residual) {
      const float r = (float)e.residual[(int64_t)m * N + n];
      if (e.binary_op == 1) v += r;
      if (e.binary_op == 2) v *= r;
    }
    if (e.unary_op == 1) v = v > 0.0f ? v : 0.0f;
    return (half_t)v;
  }
  // what is left to do after the activation pass (or all of it, where there is none), for 8 consecutive columns n .. n+7
  __device__ half8_t apply8(const float (&v)[8], int m, int n) const {
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = v[i];
    if (!activates()) {
      if (e.bias) {
        const half8_t b = *reinterpret_cast<const half8_any_t*>(e.bias + (e.bias_stride ? (int64_t)m * e.bias_stride + n : n));
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] += (float)b[i];
      }
      if (e.activation == 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = f[i] > 0.0f ? f[i] : 0.0f;
      }
    }
    if (e.residual) {
      const half8_t r = *reinterpret_cast<const half8_any_t*>(e.residual + (int64_t)m * N + n);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (e.binary_op == 1) f[i] += (float)r[i];
        if (e.binary_op == 2) f[i] *= (float)r[i];
      }
    }
    half8_t h;
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = (half_t)((e.unary_op == 1 && !(f[i] > 0.0f)) ? 0.0f : f[i]);
    return h;
  }
};
#endif

}  // namespace wq
#endif  // RELAX_AMD_CSRC_INTB_COMMON_H_
