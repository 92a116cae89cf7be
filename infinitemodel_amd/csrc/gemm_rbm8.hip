// The int8 register-B GEMM at every tile height (rbm_launch.h).
#include "rbm_launch.h"

namespace imq {
int rbm_run8(const RbArgs& a, RbmPlan p, int sdt, bool tiled, void* ws, hipStream_t st) {
  return rbm_run<8>(a, p, sdt, tiled, ws, st);
}
}  // namespace imq
