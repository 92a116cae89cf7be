// The short-batch GEMM (16 < M <= 64, int8 from 5 rows): weights dequantized in registers, K split over the waves of a
// workgroup. One translation unit per weight format (gemm_wk4.hip, gemm_wk2.hip, gemm_wk8.hip); plan and
// dispatch in gemm_wk.hip.
//
// y[M, N] = x[M, K] . dequant(W[N, K])^T, the contract, weight rounding and operand layouts of
// rb_kernel.h: a lane's 32 consecutive codes of a 64-code K step feed four v_mfma_f32_32x32x16_bf16
// slices of one 32-column block.
//
// What bounds these calls is the weight stream and how much of it is in flight, not the matrix
// cores: at 32 rows a weight byte feeds 128 flops. So
//   * a workgroup owns 32 JB columns and all (or one of `splits` ranges) of K; its 8 waves take every
//     eighth K step and run free of each other -- no barrier in the loop, P steps of weights and
//     activations in flight per wave;
//   * every wave reads the activations of its own K steps only, whole 128-byte lines of a row, and turns
//     them into A fragments through LDS it shares with no other wave (in order within the wave);
//   * scale and zero are staged once per workgroup as (bf16 s | bf16 z << 16) dwords per group and column;
//   * the waves' fp32 sums meet in LDS at the end, one 32-column block at a time, summed in wave order:
//     no partials in memory and no second launch unless there are too few column tiles for the CUs
//     (then `splits` fp32 planes and the ordered sum, as the other GEMMs).
// us per linear at M = 32 under graph replay, LDS-dequant GEMM (128-row tiles, K splits) before -> this:
// int4 4096 -> 28672 59 -> 23.4, 14336 -> 4096 33.5 -> 16.8, 4096 -> 6144 21 -> 10.1, 4096 -> 4096 15 -> 9.1;
// int8 4096 -> 14336 28 -> 17.5; int2 8192 -> 28672 125 -> 42. At M = 64: 56 -> 35, 35 -> 21, 24 -> 14,
// 18 -> 12. The VALU unpack (19 instructions per 8 codes) and the stream co-limit it: 62 MB in 23 us.
// Activations are re-read once per column tile (from L2): JB widens the tile until that traffic is below
// the weights' own, as far as the accumulators (16 IB JB) leave room for the loads in flight.
#pragma once
#include "rb_kernel.h"

namespace imq {

struct WkArgs {
  const uint16_t* x;
  int64_t sxm;
  int M, K;
  const uint8_t* q;
  int64_t sqn;
  const void* sc;
  int64_t ssn, ssg;
  const void* zr;
  int64_t szn, szg;
  int sdt, zdt;
  int N, gsh;
  uint16_t* y;
  int64_t sym;
  int tiles_n, splits, kps;
  float* part;
};

// 32 jb columns per workgroup, `splits` K ranges.
struct WkPlan {
  int jb, splits;
};

namespace {

constexpr int WK_WAVES = 8;

// Element of a scale / zero array, its dtype known at run time (uniform): raw bits, converted apart from
// the load.
IMQ_DEV uint32_t wk_raw(const void* p, int dt, int64_t i) {
  return dt == IMQ_DT_FP32 ? ((const uint32_t*)p)[i] : (uint32_t)((const uint16_t*)p)[i];
}
IMQ_DEV float wk_f32(uint32_t r, int dt) {
  return dt == IMQ_DT_FP32 ? __uint_as_float(r) : dt == IMQ_DT_FP16 ? f16_bits_to_f32(r) : bf16_bits_to_f32(r);
}

// Dwords per group of the staged pairs: the stores of 64 lanes (TPC groups x 64 / TPC columns) fall on
// distinct banks.
constexpr int wk_szs(int jb) { return 32 * jb + (jb == 4 ? 16 : jb == 2 ? 8 : 4); }
// Column blocks summed per pass: all threads have a quad when a pass holds 64 rows x 32 columns.
constexpr int wk_rj(int ib, int jb) { return ib == 1 && jb > 1 ? 2 : 1; }

// LDS bytes: the waves' activation steps (reused by the sums), then the scale / zero pairs of the
// groups a range of kps K steps touches (one more when ranges start inside a group).
inline size_t wk_lds_bytes(int bits, int ib, int jb, int kps, int gsh, int waves = WK_WAVES) {
  const size_t groups = bits == 8 ? 0 : (size_t)((((int64_t)kps * RB_BK) >> gsh) + 2);
  return (size_t)waves * ib * wk_rj(ib, jb) * 4096 + groups * wk_szs(jb) * 4;
}

// The outputs of a wave's 32 columns whose folded sum is not finite, again, weight by weight as the generic kernel
// sums them (generic_gemv, gemv.hip): s sum(c x) - z s sum(x) is infinity less infinity for an infinite
// activation, whose own product (c - z) s x has a sign. Lane (column n, half h) holds rows m8 + 4 h + e; bit e of
// `bad` asks for one. Only K steps with an infinite or NaN activation decide, found by the wave together; a row
// without any (a finite sum that overflowed) takes every step. Reached by non-finite sums only, and a call of its
// own on the kernel's arguments in memory, so that it takes no registers from the loop.
typedef const __attribute__((address_space(4))) WkArgs* WkKernarg;
template <int BITS>
__device__ __attribute__((noinline)) void wk_exact(WkKernarg ap, int m8, int n, uint32_t bad) {
  const WkArgs a = *(const WkArgs*)ap;
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const uint8_t* q = a.q + (int64_t)n * a.sqn;
  const int KT = a.K / RB_BK;
#pragma unroll 1
  for (int r = 0; r < 8; ++r) {
    const bool mine = (r >> 2) == h && ((bad >> (r & 3)) & 1u) != 0;
    if (__ballot(mine) == 0) continue;
    const uint16_t* x = a.x + (int64_t)(m8 + r) * a.sxm;
    float acc = 0.f;
    bool found = false, live = true;
#pragma unroll 1
    for (int pass = 0; pass < 2 && !found; ++pass) {
#pragma unroll 1
      for (int k0 = 0; k0 < KT && live; k0 += 64) {
        bool odd = false;
        if (k0 + lane < KT) {
#pragma unroll 1
          for (int c8 = 0; c8 < RB_BK / 8; ++c8) {
            const u32x4_t xv = *(const u32x4_t*)(x + (k0 + lane) * RB_BK + 8 * c8);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              const uint32_t xd = xv[d];
              odd |= (xd & 0x7f80u) == 0x7f80u || (xd & 0x7f800000u) == 0x7f800000u;
            }
          }
        }
        uint64_t steps = __ballot(odd);
        found |= steps != 0;
        if (pass == 1) steps = __ballot(k0 + lane < KT);
#pragma unroll 1
        for (; steps != 0 && live; steps &= steps - 1) {
          const int k = (k0 + __builtin_ctzll(steps)) * RB_BK;
          const int64_t g = k >> a.gsh;
          const float s = round_bf16(wk_f32(wk_raw(a.sc, a.sdt, n * a.ssn + g * a.ssg), a.sdt));
          const float z = round_bf16(wk_f32(wk_raw(a.zr, a.zdt, n * a.szn + g * a.szg), a.zdt));
#pragma unroll 1
          for (int c8 = 0; c8 < RB_BK / 8; ++c8) {
            const u32x4_t xv = *(const u32x4_t*)(x + k + 8 * c8);
            const uint32_t w = BITS == 4 ? *(const uint32_t*)(q + (k + 8 * c8) / 2) : *(const uint16_t*)(q + (k + 8 * c8) / 4);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const uint32_t xd = xv[i >> 1];
              const float c = (float)((w >> (BITS * i)) & ((1u << BITS) - 1u));
              acc = fmaf(bf16_bits_to_f32((i & 1) ? xd >> 16 : xd & 0xffffu), (c - z) * s, acc);
            }
          }
          live = __ballot(mine && acc == acc) != 0;   // a NaN stays one
        }
      }
    }
    if (mine) a.y[(int64_t)(m8 + r) * a.sym + n] = (uint16_t)cvt_pk_bf16(acc, 0.f);
  }
}

// PA: steps of activations in flight per wave (1 or 2; of weights two); MINW: waves per SIMD the registers are
// bounded for.
// FOLD (M <= 16, groups of 64 codes or more): the decode rows' arithmetic, no weight rounded: B holds the
// codes themselves, a step's sums start from zero and are folded into the total with the step's scale, and
// the zero point comes in through the rows' sums (an MFMA against ones): sum s (c - z) x = s (sum c x) -
// z s (sum x).
template <int BITS, int IB, int JB, bool TL, int PA, int MINW, int WAVES = WK_WAVES, bool FOLD = false>
__global__ __launch_bounds__(64 * WAVES, MINW) void gemm_wk_kernel(WkArgs a) {
  constexpr int PW = 2;
  static_assert(PW % PA == 0, "rings");
  static_assert(!FOLD || (IB == 1 && BITS != 8), "folded form: up to 16 rows of a group format");
  constexpr int BK = RB_BK, BN = 32 * JB, NTHR = 64 * WAVES;
  constexpr int XC = FOLD ? 2 : 4 * IB;            // 16-byte activation loads per lane per step (8 rows each)
  constexpr int SZS = wk_szs(JB), RJ = wk_rj(IB, JB);
  constexpr int QV = BITS == 8 ? 2 : 1, QB = 4 * BITS;
  using QT = std::conditional_t<BITS == 2, u32x2_t, u32x4_t>;
  extern __shared__ __align__(16) char wk_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c = lane & 31;
  const int split = blockIdx.x / a.tiles_n;
  const int n0 = (blockIdx.x - split * a.tiles_n) * BN;
  const int kt0 = split * a.kps;
  const int KT = min(a.K / BK - kt0, a.kps);       // >= 1 (the plan leaves no empty range)
  const int steps = KT > wave ? (KT - wave + WAVES - 1) / WAVES : 0;
  char* const Aw = wk_lds + wave * (IB * RJ * 4096);   // this wave's activation step, [32 IB rows][64] bf16
  uint32_t* const SZ = (uint32_t*)(wk_lds + WAVES * IB * RJ * 4096);

  // ---- load plan: offsets from the tile's first row, fixed for the whole loop; the step's part is
  // uniform. Rows past M repeat row M - 1, columns past N column N - 1 (never stored). --------------
  uint32_t xo[XC], xl[XC];
#pragma unroll
  for (int j = 0; j < XC; ++j) {
    const int row = 8 * j + (lane >> 3), ch = lane & 7;
    xo[j] = 2 * ((uint32_t)(min(row, a.M - 1) * (int)a.sxm) + ch * 8);
    xl[j] = 2 * rb_swz(row, ch);
  }
  uint32_t qo[JB];
#pragma unroll
  for (int j = 0; j < JB; ++j) {
    const int rr = min(n0 + 32 * j + c, a.N - 1) - n0;
    if constexpr (TL) {   // see rb_kernel.h: one offset, the step's slot bit xored in
      const int hr = (rr >> 3) & 1;
      qo[j] = (uint32_t)((rr >> 4) * 16 * (int)a.sqn + 1152 * hr + 16 * (rr & 7) +
                         (BITS == 8 ? 512 : BITS == 4 ? 256 : 8) * h);
    } else {
      qo[j] = (uint32_t)(rr * (int)a.sqn + QB * h);
    }
  }
  const __amdgpu_buffer_rsrc_t xrs = rb_rsrc(a.x);
  const __amdgpu_buffer_rsrc_t qrs = rb_rsrc(a.q + (int64_t)n0 * a.sqn);

  u32x4_t xr[PA][XC];
  QT qr[PW][JB][QV];
  auto kt_of = [&](int i) { return kt0 + min(wave, KT - 1) + WAVES * max(min(i, steps - 1), 0); };
  auto load_a = [&](auto setc, int i) {
    const int kt = kt_of(i);
#pragma unroll
    for (int j = 0; j < XC; ++j) xr[decltype(setc)::value % PA][j] = rb_bload128(xrs, xo[j], kt * (BK * 2));
  };
  auto load_b = [&](auto setc, int i) {
    const int kt = kt_of(i);
#pragma unroll
    for (int j = 0; j < JB; ++j)
#pragma unroll
      for (int v = 0; v < QV; ++v) {
        uint32_t vo, so;
        if constexpr (TL) {
          vo = (qo[j] ^ (((BITS == 8 ? kt : BITS == 4 ? (kt >> 1) : (kt >> 2)) & 1) << 7)) + 256 * v;
          so = BITS == 8 ? 2048 * (kt >> 1) : BITS == 4 ? 2048 * (kt >> 2) + 512 * (kt & 1)
                                                        : 2048 * (kt >> 3) + 256 * (kt & 3);
        } else {
          vo = qo[j] + 16 * v;
          so = kt * (BK * BITS / 8);
        }
        if constexpr (BITS == 2) qr[decltype(setc)::value][j][v] = rb_bload64(qrs, vo, so);
        else qr[decltype(setc)::value][j][v] = rb_bload128(qrs, vo, so);
      }
  };

  // the ring's first loads, then scale / zero: 64 x 8 / BN threads a column, each on every TPC-th group
  // of it, batches of 8 (the staging's address arithmetic runs under the ring's latency)
  auto fill = [&](auto setc) {
    if constexpr (decltype(setc)::value < PA) load_a(setc, decltype(setc)::value);
    load_b(setc, decltype(setc)::value);
    __builtin_amdgcn_sched_barrier(0);
  };
  fill(std::integral_constant<int, 0>{});
  fill(std::integral_constant<int, 1>{});
  const int g_lo = (kt0 * BK) >> a.gsh;
  if constexpr (BITS != 8) {
    constexpr int TPC = NTHR / BN, SB = 8;
    const int ngr = (((kt0 + KT) * BK - 1) >> a.gsh) - g_lo + 1;
    const int col = tid / TPC, part = tid % TPC;
    const int64_t n = min(n0 + col, a.N - 1);
    const int64_t sb = n * a.ssn + g_lo * a.ssg, zb = n * a.szn + g_lo * a.szg;
    for (int g0 = part; g0 < ngr; g0 += SB * TPC) {
      uint32_t sv[SB], zv[SB];
#pragma unroll
      for (int u = 0; u < SB; ++u) {
        const int g = min(g0 + u * TPC, ngr - 1);
        sv[u] = wk_raw(a.sc, a.sdt, sb + g * a.ssg);
        zv[u] = wk_raw(a.zr, a.zdt, zb + g * a.szg);
      }
#pragma unroll
      for (int u = 0; u < SB; ++u) {
        const int g = g0 + u * TPC;
        const float s_ = round_bf16(wk_f32(sv[u], a.sdt)), z_ = round_bf16(wk_f32(zv[u], a.zdt));
        if (g < ngr) SZ[g * SZS + col] = (__float_as_uint(s_) >> 16) | (__float_as_uint(z_) & 0xffff0000u);
      }
    }
    lds_barrier();
  }

  f32x16_t acc[IB][JB];
#pragma unroll
  for (int i = 0; i < IB; ++i)
#pragma unroll
    for (int j = 0; j < JB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  int aoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = 2 * rb_swz(c, 4 * h + s);   // bytes; + 32 rows (4096 bytes) per i

  auto step = [&](auto setc, int i) {
    constexpr int set = decltype(setc)::value;
    const int kt = kt_of(i);
#pragma unroll
    for (int j = 0; j < XC; ++j) *(u32x4_t*)(Aw + xl[j]) = xr[set % PA][j];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the step's rows visible to the wave's lanes
    float s_[JB], nz[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      s_[j] = nz[j] = 0.f;
      if constexpr (BITS != 8) {
        const uint32_t p = SZ[(((kt * BK + 32 * h) >> a.gsh) - g_lo) * SZS + 32 * j + c];
        s_[j] = __uint_as_float(p << 16);
        nz[j] = -__uint_as_float(p & 0xffff0000u) * s_[j];
      }
    }
    load_a(setc, i + PA);
    f32x16_t part[FOLD ? JB : 1], xs;                        // FOLD: the step's sums of c x and of x
    if constexpr (FOLD) {
      const uint32_t one2 = 0x3f803f80u;
      const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, u32x4_t{one2, one2, one2, one2});
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bf16x8_t af = *(const bf16x8_t*)(Aw + aoff[s]);
        xs = mfma32x32x16(af, ones, s == 0 ? f32x16_t{} : xs);
#pragma unroll
        for (int j = 0; j < JB; ++j) {
          const u32x4_t d = codes8_bf16<BITS>(qr[set][j][0][BITS == 4 ? s : s >> 1], s & 1);
          part[j] = mfma32x32x16(af, __builtin_bit_cast(bf16x8_t, d), s == 0 ? f32x16_t{} : part[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < JB; ++j)
#pragma unroll
        for (int r = 0; r < 8; ++r) acc[0][j][r] = fmaf(nz[j], xs[r], fmaf(s_[j], part[j][r], acc[0][j][r]));   // rows < 16
    }
#pragma unroll
    for (int s = 0; s < (FOLD ? 0 : 4); ++s) {
      bf16x8_t af[IB];
#pragma unroll
      for (int b = 0; b < IB; ++b) af[b] = *(const bf16x8_t*)(Aw + aoff[s] + b * 4096);
#pragma unroll
      for (int j = 0; j < JB; ++j) {
        u32x4_t d;
        if constexpr (BITS == 8) d = rb_convert8(qr[set][j][s >> 1][2 * (s & 1)], qr[set][j][s >> 1][2 * (s & 1) + 1]);
        else if constexpr (BITS == 2) d = dequant8_bf16<2>(qr[set][j][0][s >> 1], s & 1, s_[j], nz[j]);
        else d = dequant8_bf16<4>(qr[set][j][0][s], 0, s_[j], nz[j]);
        const bf16x8_t bf = __builtin_bit_cast(bf16x8_t, d);
#pragma unroll
        for (int b = 0; b < IB; ++b) acc[b][j] = mfma32x32x16(af[b], bf, acc[b][j]);
      }
    }
    load_b(setc, i + PW);
    __builtin_amdgcn_wave_barrier();                         // the rows are overwritten by the next step
    __builtin_amdgcn_sched_barrier(0);
  };
  int i = 0;
  for (; i + PW <= steps; i += PW) {
    step(std::integral_constant<int, 0>{}, i);
    step(std::integral_constant<int, 1>{}, i + 1);
  }
  if (i < steps) step(std::integral_constant<int, 0>{}, i);

  uint32_t bad = 0;                                          // FOLD: the thread's outputs that are not finite
  // ---- the waves' sums, RJ 32-column blocks at a time: a wave writes them where its activations were,
  // 16 bytes (4 rows) per lane; a thread adds the 8 waves' quads in wave order ----------------------
#pragma unroll
  for (int j = 0; j < JB; j += RJ) {
    if (j > 0) lds_barrier();
#pragma unroll
    for (int u = 0; u < RJ; ++u)
#pragma unroll
      for (int b = 0; b < IB; ++b)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          *(f32x4_t*)(Aw + (((u * IB + b) * 4 + r4) * 64 + lane) * 16) = f32x4_t{
              acc[b][j + u][4 * r4], acc[b][j + u][4 * r4 + 1], acc[b][j + u][4 * r4 + 2], acc[b][j + u][4 * r4 + 3]};
    lds_barrier();
#pragma unroll
    for (int q = tid; q < RJ * IB * 256; q += NTHR) {
      const int u = q / (IB * 256), b = (q >> 8) % IB, r4 = (q >> 6) & 3, l = q & 63;
      f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += *(const f32x4_t*)(wk_lds + w * (IB * RJ * 4096) + q * 16);
      const int n = n0 + 32 * (j + u) + (l & 31), m0 = 32 * b + 8 * r4 + 4 * (l >> 5);
      if (n >= a.N) continue;
      if (a.splits > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (m0 + e < a.M) a.part[((size_t)split * a.M + m0 + e) * a.N + n] = v[e];
      } else {
        float s8 = 1.f;
        if constexpr (BITS == 8) s8 = wk_f32(wk_raw(a.sc, a.sdt, (int64_t)n * a.ssn), a.sdt);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (m0 + e < a.M) {
            a.y[(int64_t)(m0 + e) * a.sym + n] = (uint16_t)cvt_pk_bf16(v[e] * s8, 0.f);
            if constexpr (FOLD) bad |= __builtin_isfinite(v[e]) ? 0u : 1u << e;
          }
      }
    }
  }
  if constexpr (FOLD) {                                      // one pass: wave w's lanes hold rows 8 w + 4 h + e of column c
    static_assert(JB == 1 && RJ == 1, "one quad per thread");
    if (__ballot(bad != 0) != 0) wk_exact<BITS>((WkKernarg)__builtin_amdgcn_kernarg_segment_ptr(), 8 * wave, min(n0 + c, a.N - 1), bad);
  }
}

template <int BITS, int IB, int JB, bool TL>
int wk_launch(const WkArgs& a, hipStream_t st) {
  // Two steps of weights in flight, one or two of activations, and four waves per SIMD where the
  // accumulators allow it: deeper rings at two waves per SIMD measured slower (4096 -> 28672 int4 at
  // M = 32, 64 columns: 22.3 us at 2 / 2 / 4, 28.6 at 4 / 4 / 2), a step's own chain (LDS, unpack,
  // MFMA) being as long as its loads.
  constexpr int PA = IB == 1 && JB == 2 ? 2 : 1, MINW = IB == 1 && JB <= 2 ? 4 : 2;
  const size_t lds = wk_lds_bytes(BITS, IB, JB, a.kps, a.gsh);
  auto kern = gemm_wk_kernel<BITS, IB, JB, TL, PA, MINW>;
  if (lds > 65536) {
    static int attr_set = 0;   // benign race: every caller sets the same value
    if (!__atomic_load_n(&attr_set, __ATOMIC_ACQUIRE)) {
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         device_info().max_lds);
      if (e != hipSuccess) return (int)e;
      __atomic_store_n(&attr_set, 1, __ATOMIC_RELEASE);
    }
  }
  kern<<<dim3((unsigned)(a.tiles_n * a.splits)), dim3(64 * WK_WAVES), lds, st>>>(a);
  IMQ_LAUNCH_CHECK();
  return IMQ_OK;
}

// The folded form: decode rows whose K no line or K-split kernel takes. us, generic kernel (one wave per row,
// a code at a time) -> this: int2 12096 -> 1344 M = 1 / 7 / 16 113 / 221 / 385 -> 15, 3520 -> 2560 41 / 74 / 116 ->
// 9; bound by its 12 K steps per wave in turn. One 32-column block per workgroup, 16 waves (decode shapes are short of workgroups,
// not of columns), K unsplit.
constexpr int WKD_WAVES = 16;
template <int BITS>
int wkd_launch(const WkArgs& a, hipStream_t st) {
  const size_t lds = wk_lds_bytes(BITS, 1, 1, a.kps, a.gsh, WKD_WAVES);
  // int2 fits the registers of five waves per SIMD: the next workgroup's 16 waves start once the waves without outputs
  // have ended (at four, 64 -> 152064 M = 4 94 us against 82)
  auto kern = gemm_wk_kernel<BITS, 1, 1, false, 2, BITS == 2 ? 5 : 4, WKD_WAVES, true>;
  if (lds > 65536) {
    static int attr_set = 0;   // benign race: every caller sets the same value
    if (!__atomic_load_n(&attr_set, __ATOMIC_ACQUIRE)) {
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         device_info().max_lds);
      if (e != hipSuccess) return (int)e;
      __atomic_store_n(&attr_set, 1, __ATOMIC_RELEASE);
    }
  }
  kern<<<dim3((unsigned)a.tiles_n), dim3(64 * WKD_WAVES), lds, st>>>(a);
  IMQ_LAUNCH_CHECK();
  return IMQ_OK;
}

template <int BITS, bool TL>
int wk_shape(const WkArgs& a, int jb, hipStream_t st) {
  if (a.M <= 32) {
    if (jb == 1) return wk_launch<BITS, 1, 1, TL>(a, st);
    if (jb == 2) return wk_launch<BITS, 1, 2, TL>(a, st);
    if constexpr (BITS != 8)
      if (jb == 4) return wk_launch<BITS, 1, 4, TL>(a, st);
  } else {
    if (jb == 1) return wk_launch<BITS, 2, 1, TL>(a, st);
    if (jb == 2) return wk_launch<BITS, 2, 2, TL>(a, st);
  }
  return IMQ_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace imq
