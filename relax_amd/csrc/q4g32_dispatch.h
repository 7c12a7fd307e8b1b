// Format A kernels that only wq_q4g32_linear chooses (no entry points of their own).
#ifndef RELAX_AMD_CSRC_Q4G32_DISPATCH_H_
#define RELAX_AMD_CSRC_Q4G32_DISPATCH_H_

#include "wq_host.h"

namespace wq {

// The small-batch kernel for 1 .. 64 rows under K % 64 == 32 (q4g32_skinny.hip).  N must be even: the aligned pair
// that holds the last scale of an odd number of odd rows would end past S.  Up to 8 rows the weights are not rounded
// to fp16.
inline bool q4g32_half_step_rows_ok(const uint16_t* x, int64_t N) { return N > 0 && N % 2 == 0 && aligned16(x); }
int q4g32_half_step_rows(const uint32_t* W, const uint16_t* S, const uint16_t* x, const uint16_t* bias,
                         const uint16_t* residual, uint16_t* y, int64_t M, int64_t N, int64_t K,
                         hipStream_t stream);

}  // namespace wq
#endif  // RELAX_AMD_CSRC_Q4G32_DISPATCH_H_
