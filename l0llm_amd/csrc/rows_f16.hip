// Instantiations of the multi-row weight-streaming kernel for L0H_F16 weights (see rows_kernel.h).
#include "rows_kernel.h"

namespace l0h {
int gemv_rows_f16(hipStream_t s, const GemvParams& p, int pos0) { return dispatch_rows_wt<L0H_F16>(s, p, pos0); }
}  // namespace l0h
