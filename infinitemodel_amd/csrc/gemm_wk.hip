// The short-batch GEMM (gemm_wk.h): plan and dispatch.
#include "gemm_wk.h"
#include "splitk_sum.h"

#include <algorithm>

namespace imq {

int wk_run4(const WkArgs& a, int jb, bool tiled, hipStream_t st);
int wk_run2(const WkArgs& a, int jb, bool tiled, hipStream_t st);
int wk_run8(const WkArgs& a, int jb, bool tiled, hipStream_t st);
int wkd_run2(const WkArgs& a, hipStream_t st);
int wkd_run4(const WkArgs& a, hipStream_t st);
double gemm_lds_us(int bits, int64_t M, int64_t N, int64_t K, int cus, bool planes);

namespace {

// The scale groups are powers of two >= 32 codes (int8: one per row, no shift).
int wk_gsh(int bits, int64_t G) {
  int gsh = 0;
  if (bits != 8)
    while ((1ll << gsh) < G) ++gsh;
  return gsh;
}

// Column blocks and K ranges of a call, the cheapest by a model fitted to a sweep of both over int4 / int8 /
// int2 linears of 2944 to 28672 columns and 768 to 28672 codes (it picks the measured best or one within
// 4% of it): a wave's steps cost 0.8 / 1.4 / 2.4 us at 1 / 2 / 4 column blocks (32 rows; 1.35 / 2.1 at 64)
// while the workgroups fit the CUs and in proportion to their number past that; a split costs the
// sum's launch (4.5 us with its gap) and its fp32 planes (written and read). 4096 -> 28672: 4 blocks, whole K; 14336 ->
// 4096: 2 blocks, 4 ranges (16.8 us against 18.7 for 1 block in 2); 4096 -> 4096: 1 block, whole K.
bool wk_plan(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, int max_lds, int max_splits, WkPlan* p) {
  const int ib = M <= 32 ? 1 : 2, KT = (int)(K / RB_BK), gsh = wk_gsh(bits, G);
  double best = 0;
  p->splits = 0;
  for (int jb = 1; jb <= (ib == 1 && bits != 8 ? 4 : 2); jb *= 2) {
    const int64_t T = imq_cdiv(N, 32 * jb);
    for (int s = 1; s <= max_splits; ++s) {
      const int kps = (KT + s - 1) / s;
      if (s > 1 && ((s - 1) * kps >= KT || kps < 2 * WK_WAVES || T * s > 2 * cus)) break;
      if (wk_lds_bytes(bits, ib, jb, kps, gsh) > (size_t)max_lds) continue;
      const double per = ib == 1 ? (jb == 1 ? 0.8 : jb == 2 ? 1.4 : 2.4) : (jb == 1 ? 1.35 : 2.1);
      const double fill = (double)(T * s) / cus;
      const double us = (fill > 1 ? fill : 1) * ((kps + WK_WAVES - 1) / WK_WAVES) * per +
                        (s > 1 ? 4.5 + 8e-6 / 4 * s * M * N : 0);
      if (p->splits == 0 || us < best) {
        best = us;
        *p = WkPlan{jb, s};
      }
    }
  }
  return p->splits != 0;
}

// The row counts the form takes. int4 / int2: 17 to 64 (decode rows round no weight). int8, whose integers
// are exact in bf16: from 5, where the skinny kernel restages the activations for every 16 rows of
// weights -- us, skinny -> this at M = 5 / 16: 4096 -> 4096 10.3 / 13.6 -> 8.8 / 8.7, 14336 -> 4096 25.9 / 37.8 ->
// 18.0 / 18.3, 4096 -> 14336 18.2 / 25.2 -> 15.8 / 16.3; at a vocabulary's width the skinny kernel's
// persistent tiles win up to 8 rows (3584 -> 152064 M = 8 100 against 116, M = 16 144 against 121), and at a short K,
// where this form's sum over its waves costs more than the whole call, while rows times K stay small (64 -> 65536
// M = 8 / 16 5.8 / 7.1 against 9.1 / 9.0, 192 -> 65536 M = 8 7.7 against 9.0, 256 -> 65536 M = 16 13 against 8).
bool wk_rows(int bits, int64_t M, int64_t N, int64_t K) {
  if (bits == 8 && M <= 16) return M > 4 && (M > 8 || N <= 65536) && (N <= 16384 || M * K > 1536);
  return M > 16 && M <= 64;
}

// Whether the plan is worth taking past 16 rows. Where the workgroups outnumber the CUs each pays its fixed cost
// (staging, the sum over its waves) in turn, and at a short K the LDS-dequant GEMM's tiles, half as many with
// stores as wide, are faster: us, LDS-dequant against this, 64 -> 131072 int4 M = 17 / 64 11 / 25 and 14 / 48, 512 -> 65536
// int4 M = 64 21 / 26, 768 -> 65536 int8 M = 64 19 / 24, but 768 -> 65536 int4 M = 17 21 / 16 and 2048 -> 65536 int4 M = 64
// 51 / 42. This form's us is a fit to graph replays of such calls (3 to 12% rms), c + rounds (f + step per K step of a
// wave + per K / 512), with a margin where the fit runs high; from three steps a wave it has been the faster at every
// width, and grids within the CUs differ by 2 us at most, at K = 64.
// int8 rows 5 to 8: two-block workgroups that just outnumber the CUs run a second round nearly empty, and the skinny
// kernel's persistent tiles are the faster while it can stage the rows: 3584 -> 18944 M = 6 / 8 18.4 / 19.5 against 21.5 / 21.8,
// 6144 -> 16896 M = 7 39.7 against 44.0; from 1.4 rounds on 3392 -> 23393 M = 7 26.0 against 25.0.
bool wk_worth(int bits, int64_t M, int64_t N, int64_t K, int cus, const WkPlan& p) {
  const int64_t W = imq_cdiv(N, 32 * p.jb);
  if (M <= 8) return !(p.jb == 2 && p.splits == 1 && W > cus && 5 * W <= 7 * cus && K >= 1024 && M * K <= 48 << 10);
  if (M <= 16 || p.splits > 1 || W <= cus || K > 2 * WK_WAVES * RB_BK) return true;
  struct Cost { double c, f, step, per; };
  const bool one = p.jb == 1;
  const Cost k = bits == 8 ? (M > 32 ? (one ? Cost{5.3, 0.33, 0, 1.13} : Cost{3.9, 2.85, 0.1, 1.3})
                                     : (one ? Cost{3.4, 0.3, 0.2, 0.4} : Cost{3.1, 0.6, 0.9, 0.35}))
                 : M > 32  ? (one ? Cost{6.9, 0.36, 0.3, 0.45} : Cost{6.0, 4.5, 0.2, 0.74})
                 : one     ? Cost{3.2, 2.2, 0.75, 0}
                 : bits == 4 ? (p.jb == 2 ? Cost{5.1, 1.95, 0.2, 0.55} : Cost{7.3, 3.3, 0.47, 1.56})
                             : (p.jb == 2 ? Cost{2.9, 3.3, 0.7, 0.46} : Cost{6.3, 1.76, 0, 1.94});
  const double steps = (double)imq_cdiv(K / RB_BK, WK_WAVES), us = k.c + (double)W / cus * (k.f + k.step * steps + k.per * K / 512);
  return us < (bits == 4 && M <= 32 ? 1.1 : bits == 8 || M <= 32 ? 1.0 : 1.05) * gemm_lds_us(bits, M, N, K, cus, true);
}

}  // namespace

// The short-batch GEMM's plan of an M x N x K call (int8 when G is 0) on a device of `cus` CUs, without a
// device: out = {takes the call, 32-column blocks per workgroup, K ranges}.
void wk_plan_query(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, int max_lds, int64_t* out) {
  WkPlan p{0, 0};
  const bool takes = wk_rows(bits, M, N, K) && K % RB_BK == 0 && wk_plan(bits, M, N, K, G, cus, max_lds, 8, &p) &&
                     wk_worth(bits, M, N, K, cus, p);
  out[0] = takes ? 1 : 0;
  out[1] = takes ? p.jb : 0;
  out[2] = takes ? p.splits : 0;
}

// Bytes of split-K planes a call of this shape may use. Past 16 rows: no plan has more than 8 ranges, nor more
// than two workgroups per CU when it splits (of at least N / 128 column tiles). int8 rows 5 to 16: the plan's own.
int64_t wk_workspace_bytes(int64_t M, int64_t N, int64_t K, int cus) {
  if (M > 64 || N <= 0 || K <= 0 || K % RB_BK != 0) return 0;
  if (M <= 16) {
    WkPlan p;
    if (!wk_rows(8, M, N, K) || !wk_plan(8, M, N, K, 0, cus, device_info().max_lds, 8, &p)) return 0;
    return p.splits > 1 ? p.splits * M * N * 4 : 0;
  }
  const int64_t s = std::min<int64_t>(8, 2 * (int64_t)cus / imq_cdiv(N, 128));
  return s > 1 ? s * M * N * 4 : 0;
}

// The rows of wk_rows, K a multiple of 64; groups and strides checked by the caller (gemm_wq_any; int8 has none). Scale and
// zero of any dtype. IMQ_ERR_UNSUPPORTED for offsets beyond 32 bits or tiles no LDS holds: the
// LDS-dequant GEMM takes those. Without a large enough workspace K is not split.
int gemm_wk(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
            const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg, int zdt,
            int64_t N, int64_t G, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st, bool tiled) {
  if (!wk_rows(bits, M, N, K) || K <= 0 || K % RB_BK != 0) return IMQ_ERR_UNSUPPORTED;
  if (((uintptr_t)x & 15) || (sxm & 7) || ((uintptr_t)q & 15) || (sqn & 15)) return IMQ_ERR_UNSUPPORTED;
  if ((64 * sxm + K) * 2 > 0x7fffffff || 128 * sqn + K > 0x7fffffff) return IMQ_ERR_UNSUPPORTED;
  const DevInfo d = device_info();
  WkPlan p;
  if (!wk_plan(bits, M, N, K, G, d.cus, d.max_lds, 8, &p)) return IMQ_ERR_UNSUPPORTED;
  if (!wk_worth(bits, M, N, K, d.cus, p)) return IMQ_ERR_UNSUPPORTED;
  if (p.splits > 1 && (!ws || wsb < (int64_t)p.splits * M * N * 4 || ((uintptr_t)ws & 15)))
    if (!wk_plan(bits, M, N, K, G, d.cus, d.max_lds, 1, &p)) return IMQ_ERR_UNSUPPORTED;
  const int KT = (int)(K / RB_BK), kps = (KT + p.splits - 1) / p.splits;
  const int64_t T = imq_cdiv(N, 32 * p.jb);
  if (T * p.splits > 0x7fffff) return IMQ_ERR_UNSUPPORTED;
  WkArgs a{x, sxm, (int)M, (int)K, q, sqn, sc, ssn, ssg, zr, szn, szg, sdt, zdt, (int)N, wk_gsh(bits, G), y, sym,
           (int)T, p.splits, kps, p.splits > 1 ? (float*)ws : nullptr};
  const int rc = bits == 4   ? wk_run4(a, p.jb, tiled, st)
                 : bits == 2 ? wk_run2(a, p.jb, tiled, st)
                             : wk_run8(a, p.jb, tiled, st);
  if (rc != IMQ_OK || p.splits == 1) return rc;
  if (bits != 8) return splitk_sum<4, IMQ_DT_BF16>(a.part, p.splits, a.M, a.N, sc, ssn, y, sym, st);
  switch (sdt) {   // int8: the row scale multiplies the sum
    case IMQ_DT_BF16: return splitk_sum<8, IMQ_DT_BF16>(a.part, p.splits, a.M, a.N, sc, ssn, y, sym, st);
    case IMQ_DT_FP16: return splitk_sum<8, IMQ_DT_FP16>(a.part, p.splits, a.M, a.N, sc, ssn, y, sym, st);
    case IMQ_DT_FP32: return splitk_sum<8, IMQ_DT_FP32>(a.part, p.splits, a.M, a.N, sc, ssn, y, sym, st);
  }
  return IMQ_ERR_INVALID;
}

// Decode rows (M <= 16) the decode kernels do not take for their K: the folded form, row layout, K a multiple
// of 64, groups of 2^k >= 64 codes, any dtypes and scale strides. IMQ_ERR_UNSUPPORTED: the generic kernel's.
int gemm_wkd(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
             const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg, int zdt,
             int64_t N, int64_t G, uint16_t* y, int64_t sym, hipStream_t st) {
  if (M < 1 || M > 16 || K % RB_BK != 0 || G < RB_BK || (G & (G - 1)) != 0 || N > (1 << 30)) return IMQ_ERR_UNSUPPORTED;
  const int qa = bits == 2 ? 8 : 16;               // a lane's load
  if (((uintptr_t)x & 15) || (sxm & 7) || ((uintptr_t)q % qa) || sqn % qa) return IMQ_ERR_UNSUPPORTED;
  if ((16 * sxm + K) * 2 > 0x7fffffff || 32 * sqn + K > 0x7fffffff) return IMQ_ERR_UNSUPPORTED;
  const int gsh = wk_gsh(bits, G), KT = (int)(K / RB_BK);
  if (wk_lds_bytes(bits, 1, 1, KT, gsh, WKD_WAVES) > (size_t)device_info().max_lds) return IMQ_ERR_UNSUPPORTED;
  const WkArgs a{x, sxm, (int)M, (int)K, q, sqn, sc, ssn, ssg, zr, szn, szg, sdt, zdt, (int)N, gsh, y, sym,
                 (int)imq_cdiv(N, 32), 1, KT, nullptr};
  return bits == 4 ? wkd_run4(a, st) : wkd_run2(a, st);
}

}  // namespace imq
