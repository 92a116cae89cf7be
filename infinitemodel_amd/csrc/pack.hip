// RTN packers on the GPU, bit-identical to the CPU packers the cache compiler and the load-time
// quantizer share (shard_compile.py:50-94 pack_linear_int2 / pack_linear_int4, 170-178
// pack_linear_int8; worker_quant.py:1588-1608, 1921-1944, 511-536). They quantize a weight
// already resident on the device instead of round-tripping it through the host.
//
// Group-wise asymmetric (int4 / int2), per group of G columns of a row, K zero-padded to a
// multiple of G before the min / max (the pad takes part in them):
//   scale = clamp((max - min) / qmax, 1e-8), zero = clamp(rint(-min / scale), 0, qmax),
//   q = clamp(rint(w / scale + zero), 0, qmax),
// in fp32 with IEEE division and round-half-even, the divide and the add rounded separately;
// scale and zero are stored in W's dtype (round to nearest even). Clamps are written as compares
// so that, as in torch, a -0.0 zero point (min exactly 0) keeps its sign.
// Per-row symmetric (int8), in W's own dtype: scale = max(dt(amax|w| / 127), dt(1e-8)),
// q = clamp(rint(dt(w / scale)), -127, 127) -- the quotient is rounded to dt before rint.
#include <algorithm>
#include <type_traits>

#include "imq_common.h"

namespace {

// 8 consecutive elements of a weight row as fp32 (exact widening): two 16-byte loads for fp32, one for
// the 16-bit types.
template <int DT>
struct Raw8 {
  u32x4_t d[DT == IMQ_DT_FP32 ? 2 : 1];
};
template <int DT>
IMQ_DEV void load8(Raw8<DT>& r, const void* p, int64_t idx) {
  const u32x4_t* s = (const u32x4_t*)((const char*)p + idx * (DT == IMQ_DT_FP32 ? 4 : 2));
  r.d[0] = s[0];
  if constexpr (DT == IMQ_DT_FP32) r.d[1] = s[1];
}
template <int DT>
IMQ_DEV float get8(const Raw8<DT>& r, int e) {
  if constexpr (DT == IMQ_DT_FP32) {
    const uint32_t w = r.d[e >> 2][e & 3];
    return __uint_as_float(w);
  } else {
    const uint32_t w = r.d[0][e >> 1];
    return raw_bits_to_f32<DT>((e & 1) ? (w >> 16) : (w & 0xffffu));
  }
}
// The row's elements [k, k + 8), zero past `end`; vec: the row is 16-byte aligned (k a multiple of 8).
template <int DT>
IMQ_DEV void load8_row(Raw8<DT>& r, const void* W, int64_t row, int64_t k, int64_t end, bool vec) {
  if (vec && k + 8 <= end) {
    load8<DT>(r, W, row + k);
    return;
  }
#pragma unroll
  for (int i = 0; i < (DT == IMQ_DT_FP32 ? 8 : 4); ++i) {
    uint32_t w = 0;
    if constexpr (DT == IMQ_DT_FP32) {
      if (k + i < end) w = load_raw_bits<DT>(W, row + k + i);
    } else {
      if (k + 2 * i < end) w = load_raw_bits<DT>(W, row + k + 2 * i);
      if (k + 2 * i + 1 < end) w |= load_raw_bits<DT>(W, row + k + 2 * i + 1) << 16;
    }
    r.d[i >> 2][i & 3] = w;
  }
}

// Correctly rounded v / s from r = the correctly rounded 1 / s (Markstein's division: one Newton step
// makes v r a faithful quotient, and the exact remainder of a faithful quotient rounds it correctly):
// 5 VALU operations against the ~10 of the IEEE division sequence, whose reciprocal and scaling a
// group's elements share. Exact for s in [2^-60, 2^60] and |v| <= 2^60 (no step overflows; where a tiny
// v lets the remainder underflow the quotient is below 2^-30, which neither the add of the integer
// zero point nor the rint that follow can see); other groups take the IEEE division.
IMQ_DEV float div_by(float v, float s, float r) {
  float q = v * r;
  q = fmaf(fmaf(-q, s, v), r, q);
  return fmaf(fmaf(-q, s, v), r, q);
}
IMQ_DEV bool div_by_exact(float s, float vmax) {
  return s >= 0x1p-60f && s <= 0x1p60f && vmax <= 0x1p60f;   // false for NaN
}

// A lane holds 16 consecutive columns of one group, G / 16 neighbouring lanes a whole group, a wave
// 1024 / G groups in row-major group order (so short rows leave no lane idle). HBM-bound by design:
// two 16-byte loads and one 8- or 4-byte packed store per lane, min / max by lane exchanges inside the
// group, two divisions per group and 5 operations per element instead of an IEEE division for each
// (the kernel that gave a wave one group, two elements a lane through LDS, was bound by those
// divisions and by its 4-byte loads). 4096 -> 28672 bf16 int4: 272 -> 64 us, 4.6 TB/s of reads and
// writes (a plain device copy: 4.8).
template <int BITS, int DT, int G>
__global__ __launch_bounds__(256) void pack_g_kernel(const void* __restrict__ W, int64_t sw, uint32_t groups,
                                                     int64_t in_f, FastDiv ngd, uint8_t* __restrict__ q, int64_t sq,
                                                     void* __restrict__ sc, void* __restrict__ zr, int64_t ssn,
                                                     bool wvec, bool qvec) {
  constexpr float QMAX = (float)((1 << BITS) - 1);
  constexpr int LPG = G / 16;                          // lanes of a group
  constexpr int NB = G * BITS / 8;                     // packed bytes of a group
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  const uint32_t gid0 = t / LPG;
  const int part = (int)(t % LPG);
  const bool live = gid0 < groups;
  const uint32_t gid = live ? gid0 : groups - 1;       // past the end: repeats the last group, stores nothing
  const uint32_t n = div_fast(gid, ngd);
  const uint32_t g = gid - n * ngd.d;
  const int64_t row = (int64_t)n * sw;
  const int64_t k0 = (int64_t)g * G + part * 16;
  Raw8<DT> raw[2];
  load8_row<DT>(raw[0], W, row, k0, in_f, wvec);
  load8_row<DT>(raw[1], W, row, k0 + 8, in_f, wvec);
  float v[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = get8<DT>(raw[e >> 3], e & 7);
  float lo = v[0], hi = v[0];
#pragma unroll
  for (int e = 1; e < 16; ++e) {
    lo = fminf(lo, v[e]);
    hi = fmaxf(hi, v[e]);
  }
#pragma unroll
  for (int off = LPG / 2; off > 0; off >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, off, 64));
    hi = fmaxf(hi, __shfl_xor(hi, off, 64));
  }
  float s = (hi - lo) / QMAX;
  s = s < 1e-8f ? 1e-8f : s;
  const float r = 1.f / s;
  const bool fast = div_by_exact(s, fmaxf(fabsf(lo), fabsf(hi)));
  float z = rintf(-lo / s);                            // IEEE: keeps the -0.0 of a group whose least value is 0
  z = z < 0.f ? 0.f : z;
  z = z > QMAX ? QMAX : z;
  if (!fast) {
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = v[e] / s;
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = div_by(v[e], s, r);
  }
  // clamp(rint(t)) == rint(clamp(t)) for the integer bounds; adding 2^23 rounds to an integer (half to
  // even) and leaves it in the low mantissa bits. A NaN becomes code 0 (fmaxf returns the other operand).
  uint32_t d[BITS / 2] = {};                           // 16 codes: 2 dwords of int4, 1 of int2
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const float c = fminf(fmaxf(v[e] + z, 0.f), QMAX) + 0x1p23f;
    d[e * BITS / 32] |= (__float_as_uint(c) & ((1u << BITS) - 1u)) << (e * BITS & 31);
  }
  if (!live) return;
  uint8_t* dst = q + (int64_t)n * sq + (int64_t)g * NB + part * (2 * BITS);
  if (qvec) {
    if constexpr (BITS == 4) *(u32x2_t*)dst = u32x2_t{d[0], d[1]};
    else *(uint32_t*)dst = d[0];
  } else {
#pragma unroll
    for (int b = 0; b < 2 * BITS; ++b) dst[b] = (uint8_t)(d[b >> 2] >> (8 * (b & 3)));
  }
  if (part == 0) {
    store_from_f32<DT>(sc, (int64_t)n * ssn + g, s);
    store_from_f32<DT>(zr, (int64_t)n * ssn + g, z);
  }
}

// v_cvt_i32_f32: truncates, saturates out-of-range values, NaN -> 0.
IMQ_DEV int cvt_i32(float f) {
  int i;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(f));
  return i;
}

// LPR lanes per row (8 to 64 of a wave, or the workgroup's 256), 8 columns per lane and pass: the row's |w| max,
// then the codes. The first NV passes keep the row in registers, so rows up to 8 LPR NV columns are read once
// (longer ones re-read their tail); divisions as in pack_g_kernel, one shared reciprocal per row. 4096 -> 14336
// bf16: 39 us, 4.5 TB/s (one wave per row with 2-byte loads and a division per element: 114 us).
template <int DT, int LPR, int NV>
__global__ __launch_bounds__(256) void pack_w8_kernel(const void* __restrict__ W, int64_t sw, int64_t N,
                                                      int64_t K, int8_t* __restrict__ q, int64_t sq,
                                                      void* __restrict__ sc, int64_t ssn, bool wvec, bool qvec) {
  constexpr int64_t STEP = 8 * LPR;                    // columns of a pass
  __shared__ float part[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rl = threadIdx.x % LPR;
  const int64_t n0 = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const bool live = n0 < N;
  const int64_t n = live ? n0 : N - 1;
  const int64_t row = n * sw, kl = 8 * rl;
  Raw8<DT> raw[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) load8_row<DT>(raw[i], W, row, kl + i * STEP, K, wvec);
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(get8<DT>(raw[i], e)));
  for (int64_t k = kl + NV * STEP; k < K; k += STEP) {
    Raw8<DT> t;
    load8_row<DT>(t, W, row, k, K, wvec);
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(get8<DT>(t, e)));
  }
#pragma unroll
  for (int off = (LPR < 64 ? LPR : 64) / 2; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  if constexpr (LPR == 256) {
    if (lane == 0) part[wave] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  }
  float s = round_to<DT>(amax / 127.f);
  const float smin = round_to<DT>(1e-8f);
  s = s < smin ? smin : s;
  const float r = 1.f / s;
  const bool fast = div_by_exact(s, amax);
  auto emit = [&](auto fastc, const Raw8<DT>& w, int64_t k) {
    constexpr bool FAST = decltype(fastc)::value;
    if (k >= K || !live) return;
    uint32_t d[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = get8<DT>(w, e);
      float t = FAST ? div_by(v, s, r) : v / s;
      if constexpr (DT == IMQ_DT_BF16) t = round_bf16_hw(t);
      else t = round_to<DT>(t);
      // the instruction itself, whose results are defined where a C++ cast's are not: w / 0 saturates, and a NaN (a
      // NaN weight, or 0 / 0 at an fp16 zero row) becomes 0, as in the host cast. (A float clamp and a compare
      // before a cast: 4096 x 4096 15.8 us against 14.0.)
      int ci = cvt_i32(rintf(t));
      ci = ci < -127 ? -127 : ci > 127 ? 127 : ci;
      d[e >> 2] |= ((uint32_t)ci & 0xffu) << (8 * (e & 3));
    }
    int8_t* dst = q + n * sq + k;
    if (qvec && k + 8 <= K) {
      *(u32x2_t*)dst = u32x2_t{d[0], d[1]};
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k + e < K) dst[e] = (int8_t)(d[e >> 2] >> (8 * (e & 3)));
    }
  };
  auto codes = [&](auto fastc) {
#pragma unroll
    for (int i = 0; i < NV; ++i) emit(fastc, raw[i], kl + i * STEP);
    for (int64_t k = kl + NV * STEP; k < K; k += STEP) {
      Raw8<DT> t;
      load8_row<DT>(t, W, row, k, K, wvec);
      emit(fastc, t, k);
    }
  };
  if (fast) codes(std::true_type{});
  else codes(std::false_type{});
  if (live && rl == 0) store_from_f32<DT>(sc, n * ssn, s);
}

bool dt_ok(int d) { return d == IMQ_DT_BF16 || d == IMQ_DT_FP16 || d == IMQ_DT_FP32; }

// Rows a launch covers so that its group ids (rows * ng) and threads stay below 2^31.
int64_t rows_per_launch(int64_t per_row) {
  const int64_t r = 0x7fffff00ll / per_row;
  return r > 0 ? r : 1;
}

template <int BITS, int DT, int G>
int launch_gg(const void* W, int64_t sw, int64_t N, int64_t in_f, uint8_t* q, int64_t sq, void* sc, void* zr,
              int64_t ssn, hipStream_t st) {
  constexpr int ES = DT == IMQ_DT_FP32 ? 4 : 2, LPG = G / 16;
  const int64_t ng = (in_f + G - 1) / G;
  if (ng * LPG > 0x7fffff00ll) return IMQ_ERR_UNSUPPORTED;
  const bool wvec = ((uintptr_t)W & 15) == 0 && ((sw * ES) & 15) == 0;
  const bool qvec = ((uintptr_t)q & (2 * BITS - 1)) == 0 && (sq & (2 * BITS - 1)) == 0;
  const FastDiv ngd = fast_div((uint32_t)ng);
  const int64_t step = rows_per_launch(ng * LPG);
  for (int64_t n = 0; n < N; n += step) {
    const int64_t rows = std::min(step, N - n);
    const unsigned grid = (unsigned)((rows * ng * LPG + 255) / 256);
    pack_g_kernel<BITS, DT, G><<<grid, 256, 0, st>>>((const char*)W + n * sw * ES, sw, (uint32_t)(rows * ng), in_f, ngd,
                                                    q + n * sq, sq, (char*)sc + n * ssn * ES, (char*)zr + n * ssn * ES,
                                                    ssn, wvec, qvec);
    IMQ_LAUNCH_CHECK();
  }
  return IMQ_OK;
}

template <int BITS, int DT>
int launch_g(const void* W, int64_t sw, int64_t N, int64_t in_f, int64_t G, uint8_t* q, int64_t sq, void* sc,
             void* zr, int64_t ssn, hipStream_t st) {
  switch (G) {
    case 64: return launch_gg<BITS, DT, 64>(W, sw, N, in_f, q, sq, sc, zr, ssn, st);
    case 128: return launch_gg<BITS, DT, 128>(W, sw, N, in_f, q, sq, sc, zr, ssn, st);
    case 256: return launch_gg<BITS, DT, 256>(W, sw, N, in_f, q, sq, sc, zr, ssn, st);
  }
  return IMQ_ERR_UNSUPPORTED;
}

// As many lanes as a short row has 8-column pieces (64 columns x 100000 rows: 25 us with a wave of 2-byte loads per
// row, 40 with a wave of 16-byte loads, 8 of its lanes reading, 7 with 8 rows per wave), a wave per row
// while the row fits its registers (4096 columns), else four; NV passes cover the row where they can.
template <int DT>
int launch_w8(const void* W, int64_t sw, int64_t N, int64_t K, int8_t* q, int64_t sq, void* sc, int64_t ssn,
              hipStream_t st) {
  constexpr int ES = DT == IMQ_DT_FP32 ? 4 : 2;
  const bool wvec = ((uintptr_t)W & 15) == 0 && ((sw * ES) & 15) == 0;
  const bool qvec = ((uintptr_t)q & 7) == 0 && (sq & 7) == 0;
  const int64_t step = 1 << 22;                        // rows a launch: its threads stay below 2^31
  for (int64_t n = 0; n < N; n += step) {
    const int64_t rows = std::min(step, N - n);
    const int lpr = K <= 64 ? 8 : K <= 128 ? 16 : K <= 256 ? 32 : K <= 4096 ? 64 : 256;
    const dim3 g((unsigned)((rows * lpr + 255) / 256)), b(256);
    const void* Wn = (const char*)W + n * sw * ES;
    void* scn = (char*)sc + n * ssn * ES;
    int8_t* qn = q + n * sq;
#define IMQ_P8(L_, V_) pack_w8_kernel<DT, L_, V_><<<g, b, 0, st>>>(Wn, sw, rows, K, qn, sq, scn, ssn, wvec, qvec)
    if (lpr == 8) IMQ_P8(8, 1);
    else if (lpr == 16) IMQ_P8(16, 1);
    else if (lpr == 32) IMQ_P8(32, 1);
    else if (K <= 512) IMQ_P8(64, 1);
    else if (K <= 1024) IMQ_P8(64, 2);
    else if (K <= 2048) IMQ_P8(64, 4);
    else if (K <= 4096) IMQ_P8(64, 8);
    else if (K <= 8192) IMQ_P8(256, 4);
    else IMQ_P8(256, 8);
#undef IMQ_P8
    IMQ_LAUNCH_CHECK();
  }
  return IMQ_OK;
}

template <int BITS>
int pack_g(const void* W, int64_t sw, int wdt, int64_t N, int64_t in_f, int64_t G, void* q, int64_t sq, void* sc,
           void* zr, int64_t ssn, void* stream) {
  if (!W || !q || !sc || !zr || !dt_ok(wdt)) return IMQ_ERR_INVALID;
  if (N < 0 || in_f <= 0 || G <= 0 || sw < in_f) return IMQ_ERR_INVALID;
  const int64_t ng = (in_f + G - 1) / G;
  if (sq < ng * G * BITS / 8 || ssn < ng) return IMQ_ERR_INVALID;
  if (G != 64 && G != 128 && G != 256) return IMQ_ERR_UNSUPPORTED;
  if (N == 0) return IMQ_OK;
  if (ng > 0x7fffffff) return IMQ_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  uint8_t* qb = (uint8_t*)q;
  switch (wdt) {
    case IMQ_DT_BF16: return launch_g<BITS, IMQ_DT_BF16>(W, sw, N, in_f, G, qb, sq, sc, zr, ssn, st);
    case IMQ_DT_FP16: return launch_g<BITS, IMQ_DT_FP16>(W, sw, N, in_f, G, qb, sq, sc, zr, ssn, st);
    case IMQ_DT_FP32: return launch_g<BITS, IMQ_DT_FP32>(W, sw, N, in_f, G, qb, sq, sc, zr, ssn, st);
  }
  return IMQ_ERR_INVALID;
}

// Line-tiled layout of packed weight rows (int4 / int2 codes alike: it moves bytes): in 16-row tile
// t, the 2 KiB block of line-step l (bytes [128 l, 128 l + 128) of each row) lies at 2048 (KL t + l)
// (KL = row bytes / 128); its half h holds rows 8 h .. 8 h + 7 of the tile, and its 16-byte slot s
// (0..63) piece 4 (((s >> 3) & 1) ^ h) + (s >> 4) of row 8 h + (s & 7).
IMQ_DEV void tiled_slot_src(int h, int s, int& r, int& piece) {
  r = 8 * h + (s & 7);
  piece = 4 * (((s >> 3) & 1) ^ h) + (s >> 4);
}

// One thread per 16-byte piece of the tiled array (tile) or of the row array (untile); the write
// side is the contiguous one. Pieces are 64-bit indexed.
__global__ __launch_bounds__(256) void line_tile_kernel(const uint8_t* __restrict__ src, int64_t srs, int64_t KL,
                                                        int64_t pieces, uint8_t* __restrict__ dst) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < pieces; i += (int64_t)gridDim.x * 256) {
    const int s = (int)(i & 63), h = (int)((i >> 6) & 1);
    const int64_t blk = i >> 7, t = blk / KL, l = blk - t * KL;
    int r, piece;
    tiled_slot_src(h, s, r, piece);
    const u32x4_t v = *(const u32x4_t*)(src + (16 * t + r) * srs + 128 * l + 16 * piece);
    *(u32x4_t*)(dst + 16 * i) = v;
  }
}

__global__ __launch_bounds__(256) void line_untile_kernel(const uint8_t* __restrict__ src, int64_t KL, int64_t pieces,
                                                          uint8_t* __restrict__ dst, int64_t drs) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < pieces; i += (int64_t)gridDim.x * 256) {
    // row-order piece i: row n, line-step l, piece p (8 per line)
    const int p = (int)(i & 7);
    const int64_t rl = i >> 3, n = rl / KL, l = rl - n * KL;
    const int r = (int)(n & 15), h = r >> 3;
    const int s = (r & 7) + 8 * ((p >> 2) ^ h) + 16 * (p & 3);
    const int64_t j = (((n >> 4) * KL + l) * 2 + h) * 64 + s;
    *(u32x4_t*)(dst + n * drs + 128 * l + 16 * p) = *(const u32x4_t*)(src + 16 * j);
  }
}

int tile_args_ok(const void* a, const void* b, int64_t rs, int64_t N, int64_t row_bytes) {
  if (!a || !b || N < 0 || row_bytes <= 0 || N % 16 != 0 || row_bytes % 128 != 0 || rs < row_bytes)
    return IMQ_ERR_INVALID;
  if (((uintptr_t)a & 15) || ((uintptr_t)b & 15) || (rs & 15)) return IMQ_ERR_ALIGN;
  return IMQ_OK;
}

}  // namespace

extern "C" int imq_line_tile(const void* q_rows, int64_t q_row_stride, int64_t N, int64_t row_bytes, void* q_tiled,
                             void* stream) {
  const int rc = tile_args_ok(q_rows, q_tiled, q_row_stride, N, row_bytes);
  if (rc != IMQ_OK || N == 0) return rc;
  const int64_t pieces = N * (row_bytes / 16);
  const unsigned grid = (unsigned)std::min<int64_t>((pieces + 255) / 256, 65536);
  line_tile_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint8_t*)q_rows, q_row_stride, row_bytes / 128, pieces,
                                                           (uint8_t*)q_tiled);
  IMQ_LAUNCH_CHECK();
  return IMQ_OK;
}

extern "C" int imq_line_untile(const void* q_tiled, int64_t N, int64_t row_bytes, void* q_rows, int64_t q_row_stride,
                               void* stream) {
  const int rc = tile_args_ok(q_tiled, q_rows, q_row_stride, N, row_bytes);
  if (rc != IMQ_OK || N == 0) return rc;
  const int64_t pieces = N * (row_bytes / 16);
  const unsigned grid = (unsigned)std::min<int64_t>((pieces + 255) / 256, 65536);
  line_untile_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint8_t*)q_tiled, row_bytes / 128, pieces,
                                                             (uint8_t*)q_rows, q_row_stride);
  IMQ_LAUNCH_CHECK();
  return IMQ_OK;
}

extern "C" int imq_pack_w4(const void* W, int64_t w_row_stride, int w_dtype, int64_t N, int64_t in_features,
                           int64_t group_size, void* qweight, int64_t q_row_stride, void* scale, void* zero,
                           int64_t sz_row_stride, void* stream) {
  return pack_g<4>(W, w_row_stride, w_dtype, N, in_features, group_size, qweight, q_row_stride, scale, zero,
                   sz_row_stride, stream);
}

extern "C" int imq_pack_w2(const void* W, int64_t w_row_stride, int w_dtype, int64_t N, int64_t in_features,
                           int64_t group_size, void* qweight, int64_t q_row_stride, void* scale, void* zero,
                           int64_t sz_row_stride, void* stream) {
  return pack_g<2>(W, w_row_stride, w_dtype, N, in_features, group_size, qweight, q_row_stride, scale, zero,
                   sz_row_stride, stream);
}

extern "C" int imq_pack_w8(const void* W, int64_t w_row_stride, int w_dtype, int64_t N, int64_t K, void* qweight,
                           int64_t q_row_stride, void* scale, int64_t s_stride_n, void* stream) {
  if (!W || !qweight || !scale || !dt_ok(w_dtype)) return IMQ_ERR_INVALID;
  if (N < 0 || K <= 0 || w_row_stride < K || q_row_stride < K || s_stride_n < 1) return IMQ_ERR_INVALID;
  if (N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  int8_t* qb = (int8_t*)qweight;
  switch (w_dtype) {
    case IMQ_DT_BF16: return launch_w8<IMQ_DT_BF16>(W, w_row_stride, N, K, qb, q_row_stride, scale, s_stride_n, st);
    case IMQ_DT_FP16: return launch_w8<IMQ_DT_FP16>(W, w_row_stride, N, K, qb, q_row_stride, scale, s_stride_n, st);
    case IMQ_DT_FP32: return launch_w8<IMQ_DT_FP32>(W, w_row_stride, N, K, qb, q_row_stride, scale, s_stride_n, st);
  }
  return IMQ_ERR_INVALID;
}
