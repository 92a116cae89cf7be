// The int4 short-batch GEMM (gemm_wk.h).
#include "gemm_wk.h"

namespace imq {
int wk_run4(const WkArgs& a, int jb, bool tiled, hipStream_t st) {
  return tiled ? wk_shape<4, true>(a, jb, st) : wk_shape<4, false>(a, jb, st);
}
}  // namespace imq
