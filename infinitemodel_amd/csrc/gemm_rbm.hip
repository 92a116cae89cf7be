// Register-B GEMM (rb_kernel.h) at any tile height of 96 to 256 rows, scale and zero both bf16 or both fp16:
// plan and dispatch. M > 64.
#include "rbm_launch.h"

namespace imq {

int rbm_run4(const RbArgs& a, RbmPlan p, int sdt, bool tiled, void* ws, hipStream_t st);
int rbm_run2(const RbArgs& a, RbmPlan p, int sdt, bool tiled, void* ws, hipStream_t st);
int rbm_run8(const RbArgs& a, RbmPlan p, int sdt, bool tiled, void* ws, hipStream_t st);
void gemm_plan_query(int64_t M, int64_t N, int64_t K, int cus, int64_t* out);
double gemm_lds_us(int bits, int64_t M, int64_t N, int64_t K, int cus, bool planes);

namespace {

// Bytes of split-K planes a plan may use. Up to 512 rows, where the LDS-dequant GEMM is the alternative, the
// planes of a good plan stay in the last-level cache beside the operands (int8 14336 -> 4096 at M = 512 in 8
// planes of 8 MiB: 73.5 us against 70.3); larger batches compare with unsplit tiles on half the CUs.
constexpr int64_t rbm_max_planes(int64_t M) { return (M <= 512 ? 48ll : 64ll) << 20; }

// us of `splits` fp32 planes: the sum's launch with its gap, the planes written and read (mostly from cache).
double planes_us(int s, int64_t M, int64_t N) { return s > 1 ? 4.5 + 1e-6 * s * M * N : 0; }

// The tile plan, the cheapest by a model fitted to sweeps of heights and splits over 4096 x 4096 .. 28672 at
// M 96 .. 2048 (it picks the measured best or one within 5%): a 64-code step of an ib x 32 row, 256-column
// tile takes 0.46 + 0.163 ib us (int8 0.32 + 0.145 ib); int4 / int2 steps 15% more once K is split more than
// two ways (short ranges expose the load latency their unpack otherwise hides); heights up to 128 rows
// keep two workgroups on a CU, whose steps then overlap to 0.89 of that each. Row blocks are spread
// evenly over the row tiles (777 rows: 4 tiles of 7 blocks, not 4 of 8). Returns the modelled us.
double rbm_plan(int bits, int64_t M, int64_t N, int64_t K, int cus, bool planes, RbmPlan* p) {
  const int KT = (int)(K / RB_BK);
  const int64_t blocks = imq_cdiv(M, 32), cols = imq_cdiv(N, 256);
  double best = -1;
  const int64_t rt0 = imq_cdiv(blocks, 8);
  for (int64_t rt = rt0; rt <= 3 * rt0; ++rt) {
    const int ib = (int)imq_cdiv(blocks, rt);
    if (ib < 3) break;
    if (rt > rt0 && ib == (int)imq_cdiv(blocks, rt - 1)) continue;   // the same height with idle tiles
    const double t1 = bits == 8 ? 0.32 + 0.145 * ib : 0.46 + 0.163 * ib;
    for (int s = 1; s <= (planes ? 8 : 1); ++s) {
      const int kps = (KT + s - 1) / s;
      const int64_t W = rt * cols * s;
      if (s > 1 && ((s - 1) * kps >= KT || kps < 8 || W > 2 * (int64_t)cus || 4ll * s * M * N > rbm_max_planes(M))) break;
      const double t = bits != 8 && s > 2 ? 1.15 * t1 : t1;
      double us;
      if (W <= cus) us = kps * t;
      else if (ib <= 4) us = (double)((W + 2 * cus - 1) / (2 * cus)) * kps * 2 * 0.89 * t;
      else us = (double)((W + cus - 1) / cus) * kps * t;
      us += 3 + planes_us(s, M, N);
      if (best < 0 || us < best) {
        best = us;
        *p = RbmPlan{ib, s};
      }
    }
  }
  return best;
}

// The LDS-dequant GEMM's modelled us on the same call (its plan as gemm_plan_query gives it).
double lds_us(int64_t M, int64_t N, int64_t K, int cus, bool planes) {
  int64_t out[5] = {};
  gemm_plan_query(M, N, K, cus, out);
  const int64_t s = planes ? out[3] : 1, W = imq_cdiv(M, out[1]) * imq_cdiv(N, out[2]) * s;
  return 3 + (double)imq_cdiv(W, cus) * imq_cdiv(K / RB_BK, s) * (out[1] == 256 ? 1.1 : 0.87) + planes_us((int)s, M, N);
}

// A plan's us where its K ranges are short: the fixed cost of a tile grows with its height (the epilogue), fitted to
// graph replays at every height and M 65 .. 512 (7.5% rms; rbm_plan and lds_us are fitted to long ranges, where
// they are nearer).
double short_us(int bits, int64_t M, int64_t N, int64_t K, int cus, const RbmPlan& p) {
  const int64_t kps = imq_cdiv(K / RB_BK, p.splits), W = imq_cdiv(M, 32 * p.ib) * imq_cdiv(N, 256) * p.splits;
  const double t = 0.6 + 1.88 * p.ib + kps * (bits == 8 ? 0.21 + 0.146 * p.ib : 0.447 + 0.127 * p.ib);
  const double rounds = W <= cus ? 1 : p.ib <= 4 ? 1.72 * imq_cdiv(W, 2 * cus) : (double)imq_cdiv(W, cus);
  return 0.8 + rounds * t + (p.splits > 1 ? 1 + 1.15e-6 * p.splits * M * N : 0);
}

// The tile height a row-layout int4 or int2 call runs at, its splits kept (so its sums are the line-tiled call's bit
// for bit). A K step of such a weight is 32 or 16 bytes of each row, so a 128-byte line is read over 4 or 8 steps, and two
// workgroups to a CU lose it from the L2 between them (fetched, 11776 -> 21440 at 241 rows in 96-row tiles: 516 MB in rows,
// 234 MB line-tiled, 89 MB in rows at 256-row tiles): up to 400 workgroups 1.22 times rbm_plan's estimate,
// up to 512 1.55, past that 1.35 (means of 180 calls; line-tiled 1.0 to 1.1). us at 241 rows, three 96-row tiles against
// one of 256: int4 11648 -> 21440 360 / 181, 6848 -> 36480 345 / 200.
int rows_height(int64_t M, int64_t N, int cus, const RbmPlan& p) {
  const int64_t blocks = imq_cdiv(M, 32), cols = imq_cdiv(N, 256), rt0 = imq_cdiv(blocks, 8);
  if (p.ib > 4 || imq_cdiv(blocks, p.ib) * cols * p.splits <= cus) return p.ib;
  double best = 0;
  int height = p.ib;
  for (int64_t rt = rt0; rt <= 3 * rt0; ++rt) {
    const int ib = (int)imq_cdiv(blocks, rt);
    if (ib < 3) break;
    const int64_t W = imq_cdiv(blocks, ib) * cols * p.splits;
    const double pair = 2 * 0.89 * (5 * W <= 8 * cus ? 1.22 : W <= 2 * cus ? 1.55 : 1.35);
    const double us = (0.46 + 0.163 * ib) * (W <= cus ? 1 : ib <= 4 ? pair * imq_cdiv(W, 2 * cus) : (double)imq_cdiv(W, cus));
    if (best == 0 || us < best) {
      best = us;
      height = ib;
    }
  }
  return height;
}

// Whether this GEMM takes a call, the LDS-dequant GEMM the rest. us, LDS-dequant against this kernel, where each side
// of a line was wrong before it: 200 rows, 64 -> 152064 int4 31 / 39 and 448 -> 100000 int4 at 512 rows 87 / 106; int8
// at 96 rows, 1024 -> 4096 13.0 / 13.9 (8 steps a range); int2 at 1024 rows, 64 -> 152064 117 / 162.
bool rbm_takes(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, bool planes, RbmPlan* p) {
  if (M <= 64 || N <= 0 || K <= 0 || K % RB_BK != 0 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return false;
  if (bits != 8 && (G < 32 || (G & (G - 1)) != 0)) return false;
  const double us = rbm_plan(bits, M, N, K, cus, planes, p);
  if (us <= 0) return false;
  const double ratio = short_us(bits, M, N, K, cus, *p) / gemm_lds_us(bits, M, N, K, cus, planes);
  if (M > 512) {
    // int2 of short K and tiles for more than half of 256 CUs, or of few columns and K up to 4096: the fixed cost
    // decides (2048 -> 1024 at 985 rows 19.6 / 23.7). int4 and int8 have had a register-B form above 512 rows
    // throughout, and smaller grids differ by a microsecond at most.
    if (bits != 2) return true;
    if (K <= 512) return imq_cdiv(M, 32 * p->ib) * imq_cdiv(N, 256) <= 128 || ratio < 1.0;
    return K > 4096 || N > 1024 || ratio < 0.95;
  }
  // up to 512 rows the LDS-dequant GEMM keeps the calls the model puts within its own spread, and short ranges where
  // its fixed cost is the smaller (by more than the two fits' spread where K is only short for its splits: at 12%
  // modelled, 4 to 13% measured; below that the two are within 5% of each other)
  if (us >= 0.96 * lds_us(M, N, K, cus, planes)) return false;
  // int8 of K up to 320, or of one 128-row tile and K up to 1024, where both are within the fits' spread: the LDS-dequant
  // GEMM unless 5% is modelled (192 -> 12352 at 132 rows 8.9 / 10.1, 896 -> 256 at 79 rows 13.7 / 14.9)
  if (bits == 8 && (K <= 320 || (M <= 128 && K <= 1024))) return ratio < 0.95;
  if (imq_cdiv(K / RB_BK, p->splits) > 12) return true;
  return ratio < (K <= 512 ? 1.0 : 1.12);
}

}  // namespace

// The plan of a call without a device (workspace given): out = {takes the call, 32-row blocks per tile, K splits}.
void rbm_plan_query(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, int64_t* out) {
  RbmPlan p{0, 0};
  const bool takes = rbm_takes(bits, M, N, K, G, cus, true, &p);
  out[0] = takes ? 1 : 0;
  out[1] = takes ? p.ib : 0;
  out[2] = takes ? p.splits : 0;
}

int64_t rbm_workspace_bytes(int64_t M, int64_t N, int64_t K, int cus) {
  int64_t need = 0;
  for (int bits : {4, 8}) {                        // int2 plans as int4
    RbmPlan p;
    if (rbm_takes(bits, M, N, K, 128, cus, true, &p) && p.splits > 1) need = 4 * p.splits * M * N > need ? 4 * p.splits * M * N : need;
  }
  return need;
}

// Operands as gemm_wq_any checked them. IMQ_ERR_UNSUPPORTED: another GEMM is as fast or the layout is not
// covered (other dtype pairs, offsets beyond 32 bits).
int gemm_rbm(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
             const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg, int zdt,
             int64_t N, int64_t G, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st, bool tiled) {
  if (sdt != IMQ_DT_BF16 && sdt != IMQ_DT_FP16) return IMQ_ERR_UNSUPPORTED;
  if (bits != 8 && sdt != zdt) return IMQ_ERR_UNSUPPORTED;
  // the kernel's buffer offsets from a tile's first row (activations, weights, scale / zero)
  if ((256 * sxm + K) * 2 > 0x7fffffff || 256 * sqn + K > 0x7fffffff) return IMQ_ERR_UNSUPPORTED;
  int gsh = 0;
  if (bits != 8) {
    while ((1ll << gsh) < G) ++gsh;
    if (ssg < 0 || szg < 0 || ssn < 0 || szn < 0) return IMQ_ERR_UNSUPPORTED;
    const int64_t ng = K / G + 1;
    if ((256 * ssn + ng * ssg) * 4 > 0x7fffffff || (256 * szn + ng * szg) * 4 > 0x7fffffff) return IMQ_ERR_UNSUPPORTED;
  }
  const int cus = device_info().cus;
  RbmPlan p;
  if (!rbm_takes(bits, M, N, K, G, cus, true, &p)) return IMQ_ERR_UNSUPPORTED;
  if (p.splits > 1 && (!ws || wsb < 4 * p.splits * M * N || ((uintptr_t)ws & 15)))
    if (!rbm_takes(bits, M, N, K, G, cus, false, &p)) return IMQ_ERR_UNSUPPORTED;
  RbArgs a{x, sxm, (int)M, (int)K, q, sqn, sc, ssn, ssg, zr, szn, szg, (int)N, gsh, y, sym, 0, 0, 1, 0, nullptr};
  if (bits != 8 && !tiled) p.ib = rows_height(M, N, cus, p);
  if (bits == 4) return rbm_run4(a, p, sdt, tiled, ws, st);
  if (bits == 2) return rbm_run2(a, p, sdt, tiled, ws, st);
  return rbm_run8(a, p, sdt, tiled, ws, st);
}

}  // namespace imq
