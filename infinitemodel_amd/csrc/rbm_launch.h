// Launchers of the register-B GEMM (rb_kernel.h) at any tile height, one translation unit per weight
// format (gemm_rbm4.hip, gemm_rbm2.hip, gemm_rbm8.hip); the plan and the dispatch are in gemm_rbm.hip.
#pragma once
#include "rb_kernel.h"
#include "splitk_sum.h"

namespace imq {

// Tile plan of one call: ib 32-row blocks per workgroup tile, K split `splits` ways.
struct RbmPlan {
  int ib, splits;
};

namespace {

template <int BITS, int SDT, int IB, bool TL>
int rbm_launch(const RbArgs& a0, int splits, void* ws, hipStream_t st) {
  constexpr int NW = 4, BM = 32 * IB, BN = 64 * NW;
  // two waves per SIMD fit up to 128 rows (accumulators 32 IB registers)
  constexpr int MINW = IB <= 4 ? 2 : 1;
  RbArgs a = a0;
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = (a.N + BN - 1) / BN;
  const int64_t T = (int64_t)a.tiles_m * a.tiles_n;
  const int KT = a.K / RB_BK;
  a.kps = (KT + splits - 1) / splits;
  a.splits = splits;
  a.part = splits > 1 ? (float*)ws : nullptr;
  if (T * splits > 0x7fffffff) return IMQ_ERR_UNSUPPORTED;
  constexpr size_t lds = (size_t)3 * BM * RB_BK * 2;
  auto kern = gemm_rb_kernel<BITS, SDT, SDT, IB, NW, 0, 2, false, TL, MINW>;
  if (lds > 65536) {
    static int attr_set = 0;   // benign race: every caller sets the same value
    if (!__atomic_load_n(&attr_set, __ATOMIC_ACQUIRE)) {
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return (int)e;
      __atomic_store_n(&attr_set, 1, __ATOMIC_RELEASE);
    }
  }
  kern<<<dim3((unsigned)(T * splits)), dim3(64 * NW), lds, st>>>(a);
  IMQ_LAUNCH_CHECK();
  if (splits > 1) return splitk_sum<BITS, SDT>(a.part, splits, a.M, a.N, a.sc, a.ssn, a.y, a.sym, st);
  return IMQ_OK;
}

template <int BITS, int SDT, bool TL>
int rbm_ib(const RbArgs& a, RbmPlan p, void* ws, hipStream_t st) {
  switch (p.ib) {
    case 3: return rbm_launch<BITS, SDT, 3, TL>(a, p.splits, ws, st);
    case 4: return rbm_launch<BITS, SDT, 4, TL>(a, p.splits, ws, st);
    case 5: return rbm_launch<BITS, SDT, 5, TL>(a, p.splits, ws, st);
    case 6: return rbm_launch<BITS, SDT, 6, TL>(a, p.splits, ws, st);
    case 7: return rbm_launch<BITS, SDT, 7, TL>(a, p.splits, ws, st);
    case 8: return rbm_launch<BITS, SDT, 8, TL>(a, p.splits, ws, st);
  }
  return IMQ_ERR_UNSUPPORTED;
}

}  // namespace

// sdt: IMQ_DT_BF16 or IMQ_DT_FP16, scale and zero alike.
template <int BITS>
int rbm_run(const RbArgs& a, RbmPlan p, int sdt, bool tiled, void* ws, hipStream_t st) {
  if (sdt == IMQ_DT_BF16)
    return tiled ? rbm_ib<BITS, IMQ_DT_BF16, true>(a, p, ws, st) : rbm_ib<BITS, IMQ_DT_BF16, false>(a, p, ws, st);
  return tiled ? rbm_ib<BITS, IMQ_DT_FP16, true>(a, p, ws, st) : rbm_ib<BITS, IMQ_DT_FP16, false>(a, p, ws, st);
}

}  // namespace imq
