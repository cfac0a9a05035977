// Instantiations of the multi-row weight-streaming kernel for L0H_I8PC weights (see rows_kernel.h).
#include "rows_kernel.h"

namespace l0h {
int gemv_rows_i8(hipStream_t s, const GemvParams& p, int pos0) { return dispatch_rows_wt<L0H_I8PC>(s, p, pos0); }
}  // namespace l0h
