// The int2 register-B GEMM at every tile height (rbm_launch.h).
#include "rbm_launch.h"

namespace imq {
int rbm_run2(const RbArgs& a, RbmPlan p, int sdt, bool tiled, void* ws, hipStream_t st) {
  return rbm_run<2>(a, p, sdt, tiled, ws, st);
}
}  // namespace imq
