// The int4 short-batch GEMM (gemm_wk.h).
#include "gemm_wk.h"

namespace imq {
int wk_run4(const WkArgs& a, int jb, bool tiled, hipStream_t st) {
  return tiled ? wk_shape<4, true>(a, jb, st) : wk_shape<4, false>(a, jb, st);
}
int wkd_run4(const WkArgs& a, hipStream_t st) { return wkd_launch<4>(a, st); }
}  // namespace imq
