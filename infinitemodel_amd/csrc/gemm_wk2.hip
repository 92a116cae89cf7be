// The int2 short-batch GEMM (gemm_wk.h).
#include "gemm_wk.h"

namespace imq {
int wk_run2(const WkArgs& a, int jb, bool tiled, hipStream_t st) {
  return tiled ? wk_shape<2, true>(a, jb, st) : wk_shape<2, false>(a, jb, st);
}
int wkd_run2(const WkArgs& a, hipStream_t st) { return wkd_launch<2>(a, st); }
}  // namespace imq
