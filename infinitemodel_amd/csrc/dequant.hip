// Bit-exact reference dequant kernels (int4 g-wise, int2 g-wise, int8 per-row).
//
// These reproduce `_dequant(dtype)` of the reference modules exactly, rounding after every
// elementwise op in the output dtype (worker_quant.py:638-648, 1652-1664, 439). They serve the
// module's `_dequant` on the GPU (the naive path and the self-checks) and are the unit the
// bit-exact parity tests pin. HBM-bound (2 to 4 bytes written per code): a thread takes 8 codes, one
// 2- to 8-byte load and one or two 16-byte stores, rows and groups found by multiplication instead
// of 64-bit division, two codes rounded per v_cvt_pk_bf16_f32. 4096 -> 28672 int4 to bf16: 149
// (byte loads, element stores, two 64-bit divisions per thread) -> 57 us, 5.2 TB/s;
// int8 4096 -> 14336 112 -> 30 us.
#include <algorithm>

#include "imq_common.h"

namespace {

// fp32 values -> ODT, two per dword for the 16-bit types, round to nearest even. HW: the hardware pack
// (bit-equal to store_from_f32 for every non-NaN value).
template <int ODT, bool HW>
IMQ_DEV uint32_t pack2(float a, float b) {
  static_assert(ODT != IMQ_DT_FP32, "16-bit types");
  if constexpr (ODT == IMQ_DT_FP16) return f32_to_f16_bits(a) | (f32_to_f16_bits(b) << 16);
  else if constexpr (HW) return cvt_pk_bf16(a, b);
  else return f32_to_bf16_bits(a) | (f32_to_bf16_bits(b) << 16);
}

// 8 results: d[i] = ODT(ODT(c[i] - z) * s) (ZERO) or ODT(c[i] * s), as the dwords of the row.
template <int ODT, bool ZERO, bool HW>
IMQ_DEV void dequant_values(const float* c, float s, float z, uint32_t* o) {
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float a = c[i], b = c[i + 1];
    if constexpr (ZERO) {
      a -= z;
      b -= z;
      if constexpr (ODT != IMQ_DT_FP32) {
        const uint32_t p = pack2<ODT, HW>(a, b);
        a = raw_bits_to_f32<ODT>(p & 0xffffu);
        b = raw_bits_to_f32<ODT>(p >> 16);
      }
    }
    if constexpr (ODT == IMQ_DT_FP32) {
      o[i] = __float_as_uint(a * s);
      o[i + 1] = __float_as_uint(b * s);
    } else {
      a *= s;
      b *= s;
      // fp16: a product and its conversion would become one v_fma_mixlo_f16 that adds +0, and a zero its sign
      if constexpr (ODT == IMQ_DT_FP16) asm("" : "+v"(a), "+v"(b));
      o[i / 2] = pack2<ODT, HW>(a, b);
    }
  }
}

// The 8 results at column k of an output row (elements past `end` are not written); vec: 16-byte
// aligned rows.
template <int ODT>
IMQ_DEV void store8(void* out, int64_t row, int64_t k, int64_t end, const uint32_t* o, bool vec) {
  if (vec && k + 8 <= end) {
    u32x4_t* d = (u32x4_t*)((char*)out + (row + k) * (ODT == IMQ_DT_FP32 ? 4 : 2));
    d[0] = u32x4_t{o[0], o[1], o[2], o[3]};
    if constexpr (ODT == IMQ_DT_FP32) d[1] = u32x4_t{o[4], o[5], o[6], o[7]};
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (k + i >= end) break;
    if constexpr (ODT == IMQ_DT_FP32) ((uint32_t*)out)[row + k + i] = o[i];
    else ((uint16_t*)out)[row + k + i] = (uint16_t)(o[i >> 1] >> (16 * (i & 1)));
  }
}

// Thread t: codes [8 c, 8 c + 8) of row n, t = n * chunks + c. All 8 share one group (G is a
// multiple of 8 for every format the library accepts; checked on the host).
template <int BITS, int SDT, int ZDT, int ODT>
__global__ __launch_bounds__(256) void dequant_g_kernel(
    const uint8_t* __restrict__ q, int64_t sq, const void* __restrict__ sc, int64_t ssn, int64_t ssg,
    const void* __restrict__ zr, int64_t szn, int64_t szg, uint32_t total, int64_t in_f, FastDiv chd, FastDiv gd,
    void* __restrict__ out, int64_t so, bool qvec, bool ovec) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= total) return;
  const uint32_t n = div_fast(t, chd), c = t - n * chd.d, g = div_fast(c, gd);
  const uint8_t* qp = q + (int64_t)n * sq + (int64_t)c * BITS;
  uint32_t bits = 0;
  if (qvec) {
    if constexpr (BITS == 4) bits = *(const uint32_t*)qp;
    else bits = *(const uint16_t*)qp;
  } else {
#pragma unroll
    for (int b = 0; b < BITS; ++b) bits |= (uint32_t)qp[b] << (8 * b);
  }
  const float z = round_to<ODT>(load_as_f32<ZDT>(zr, (int64_t)n * szn + (int64_t)g * szg));
  const float s = round_to<ODT>(load_as_f32<SDT>(sc, (int64_t)n * ssn + (int64_t)g * ssg));
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)((bits >> (BITS * i)) & ((1u << BITS) - 1u));
  uint32_t o[ODT == IMQ_DT_FP32 ? 8 : 4];
  // finite scale and zero give no NaN (only overflow to infinity), which the two packs treat alike
  if (__builtin_isfinite(s) && __builtin_isfinite(z)) dequant_values<ODT, true, true>(v, s, z, o);
  else dequant_values<ODT, true, false>(v, s, z, o);
  store8<ODT>(out, (int64_t)n * so, 8ll * c, in_f, o, ovec);
}

template <int SDT, int ODT>
__global__ __launch_bounds__(256) void dequant_w8_kernel(const int8_t* __restrict__ q, int64_t sq,
                                                         const void* __restrict__ sc, int64_t ssn, uint32_t total,
                                                         int64_t K, FastDiv chd, void* __restrict__ out, int64_t so,
                                                         bool qvec, bool ovec) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= total) return;
  const uint32_t n = div_fast(t, chd), c = t - n * chd.d;
  const int8_t* qp = q + (int64_t)n * sq + 8ll * c;
  uint32_t w[2] = {0u, 0u};
  if (qvec && 8ll * c + 8 <= K) {
    const u32x2_t p = *(const u32x2_t*)qp;
    w[0] = p[0];
    w[1] = p[1];
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (8ll * c + i < K) w[i >> 2] |= (uint32_t)(uint8_t)qp[i] << (8 * (i & 3));
  }
  const float s = load_as_f32<SDT>(sc, (int64_t)n * ssn);
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)(int8_t)(w[i >> 2] >> (8 * (i & 3)));
  uint32_t o[ODT == IMQ_DT_FP32 ? 8 : 4];
  // q.to(x_dtype) is exact for |q| <= 127; one fp32 product, one rounding to the result dtype.
  if (__builtin_isfinite(s)) dequant_values<ODT, false, true>(v, s, 0.f, o);
  else dequant_values<ODT, false, false>(v, s, 0.f, o);
  store8<ODT>(out, (int64_t)n * so, 8ll * c, K, o, ovec);
}

// Rows of `chunks` threads one launch covers (its threads stay below 2^31).
inline int64_t rows_per_launch(int64_t chunks) { return std::max<int64_t>(1, 0x7fffff00ll / chunks); }

template <int DT>
constexpr int esize() { return DT == IMQ_DT_FP32 ? 4 : 2; }

template <int BITS, int SDT, int ZDT, int ODT>
int launch_g(const void* q, int64_t sq, const void* sc, int64_t ssn, int64_t ssg, const void* zr,
             int64_t szn, int64_t szg, int64_t N, int64_t in_f, int64_t G, void* out, int64_t so,
             hipStream_t st) {
  const int64_t chunks = imq_cdiv(in_f, 8);
  if (N == 0 || chunks == 0) return IMQ_OK;
  if (chunks > 0x7fffff00ll) return IMQ_ERR_UNSUPPORTED;
  constexpr int OES = esize<ODT>(), QA = BITS == 4 ? 4 : 2;
  const bool qvec = ((uintptr_t)q % QA) == 0 && sq % QA == 0;
  const bool ovec = ((uintptr_t)out & 15) == 0 && ((so * OES) & 15) == 0;
  const FastDiv chd = fast_div((uint32_t)chunks), gd = fast_div((uint32_t)std::min<int64_t>(G / 8, 0x7fffffff));
  const int64_t step = rows_per_launch(chunks);
  for (int64_t n = 0; n < N; n += step) {
    const int64_t rows = std::min(step, N - n);
    const uint32_t total = (uint32_t)(rows * chunks);
    dequant_g_kernel<BITS, SDT, ZDT, ODT><<<dim3((total + 255u) / 256u), dim3(256), 0, st>>>(
        (const uint8_t*)q + n * sq, sq, (const char*)sc + n * ssn * esize<SDT>(), ssn, ssg,
        (const char*)zr + n * szn * esize<ZDT>(), szn, szg, total, in_f, chd, gd, (char*)out + n * so * OES, so, qvec,
        ovec);
    IMQ_LAUNCH_CHECK();
  }
  return IMQ_OK;
}

template <int BITS, int SDT, int ZDT>
int dispatch_out(int odt, const void* q, int64_t sq, const void* sc, int64_t ssn, int64_t ssg,
                 const void* zr, int64_t szn, int64_t szg, int64_t N, int64_t in_f, int64_t G,
                 void* out, int64_t so, hipStream_t st) {
  switch (odt) {
    case IMQ_DT_BF16: return launch_g<BITS, SDT, ZDT, IMQ_DT_BF16>(q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
    case IMQ_DT_FP16: return launch_g<BITS, SDT, ZDT, IMQ_DT_FP16>(q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
    case IMQ_DT_FP32: return launch_g<BITS, SDT, ZDT, IMQ_DT_FP32>(q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
  }
  return IMQ_ERR_INVALID;
}

template <int BITS, int SDT>
int dispatch_z(int zdt, int odt, const void* q, int64_t sq, const void* sc, int64_t ssn, int64_t ssg,
               const void* zr, int64_t szn, int64_t szg, int64_t N, int64_t in_f, int64_t G, void* out,
               int64_t so, hipStream_t st) {
  switch (zdt) {
    case IMQ_DT_BF16: return dispatch_out<BITS, SDT, IMQ_DT_BF16>(odt, q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
    case IMQ_DT_FP16: return dispatch_out<BITS, SDT, IMQ_DT_FP16>(odt, q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
    case IMQ_DT_FP32: return dispatch_out<BITS, SDT, IMQ_DT_FP32>(odt, q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
  }
  return IMQ_ERR_INVALID;
}

template <int BITS>
int dequant_g(const void* q, int64_t sq, const void* sc, int64_t ssn, int64_t ssg, int sdt,
              const void* zr, int64_t szn, int64_t szg, int zdt, int64_t N, int64_t in_f, int64_t G,
              void* out, int64_t so, int odt, void* stream) {
  if (!q || !sc || !zr || !out || N < 0 || in_f < 0 || G <= 0 || (G % 8) != 0) return IMQ_ERR_INVALID;
  if (sq < (imq_cdiv(in_f, G) * G * BITS) / 8) return IMQ_ERR_INVALID;
  hipStream_t st = (hipStream_t)stream;
  switch (sdt) {
    case IMQ_DT_BF16: return dispatch_z<BITS, IMQ_DT_BF16>(zdt, odt, q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
    case IMQ_DT_FP16: return dispatch_z<BITS, IMQ_DT_FP16>(zdt, odt, q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
    case IMQ_DT_FP32: return dispatch_z<BITS, IMQ_DT_FP32>(zdt, odt, q, sq, sc, ssn, ssg, zr, szn, szg, N, in_f, G, out, so, st);
  }
  return IMQ_ERR_INVALID;
}

template <int SDT, int ODT>
int launch_w8(const int8_t* q, int64_t sq, const void* sc, int64_t ssn, int64_t N, int64_t K, void* out, int64_t so,
              hipStream_t st) {
  const int64_t chunks = imq_cdiv(K, 8);
  if (N == 0 || chunks == 0) return IMQ_OK;
  if (chunks > 0x7fffff00ll) return IMQ_ERR_UNSUPPORTED;
  constexpr int OES = esize<ODT>();
  const bool qvec = ((uintptr_t)q & 7) == 0 && (sq & 7) == 0;
  const bool ovec = ((uintptr_t)out & 15) == 0 && ((so * OES) & 15) == 0;
  const FastDiv chd = fast_div((uint32_t)chunks);
  const int64_t step = rows_per_launch(chunks);
  for (int64_t n = 0; n < N; n += step) {
    const int64_t rows = std::min(step, N - n);
    const uint32_t total = (uint32_t)(rows * chunks);
    dequant_w8_kernel<SDT, ODT><<<dim3((total + 255u) / 256u), dim3(256), 0, st>>>(
        q + n * sq, sq, (const char*)sc + n * ssn * esize<SDT>(), ssn, total, K, chd, (char*)out + n * so * OES, so,
        qvec, ovec);
    IMQ_LAUNCH_CHECK();
  }
  return IMQ_OK;
}

template <int SDT>
int dequant8_out(int odt, const void* q, int64_t sq, const void* sc, int64_t ssn, int64_t N, int64_t K,
                 void* out, int64_t so, hipStream_t st) {
  const int8_t* qb = (const int8_t*)q;
  switch (odt) {
    case IMQ_DT_BF16: return launch_w8<SDT, IMQ_DT_BF16>(qb, sq, sc, ssn, N, K, out, so, st);
    case IMQ_DT_FP16: return launch_w8<SDT, IMQ_DT_FP16>(qb, sq, sc, ssn, N, K, out, so, st);
    case IMQ_DT_FP32: return launch_w8<SDT, IMQ_DT_FP32>(qb, sq, sc, ssn, N, K, out, so, st);
  }
  return IMQ_ERR_INVALID;
}

}  // namespace

extern "C" int imq_dequant_w4(const void* qweight, int64_t q_row_stride, const void* scale,
                              int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                              int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                              int64_t in_features, int64_t group_size, void* out, int64_t out_row_stride,
                              int out_dtype, void* stream) {
  return dequant_g<4>(qweight, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype, zero, z_stride_n,
                      z_stride_g, z_dtype, N, in_features, group_size, out, out_row_stride, out_dtype,
                      stream);
}

extern "C" int imq_dequant_w2(const void* qweight, int64_t q_row_stride, const void* scale,
                              int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                              int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                              int64_t in_features, int64_t group_size, void* out, int64_t out_row_stride,
                              int out_dtype, void* stream) {
  return dequant_g<2>(qweight, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype, zero, z_stride_n,
                      z_stride_g, z_dtype, N, in_features, group_size, out, out_row_stride, out_dtype,
                      stream);
}

extern "C" int imq_dequant_w8(const void* qweight, int64_t q_row_stride, const void* scale,
                              int64_t s_stride_n, int s_dtype, int64_t N, int64_t K, void* out,
                              int64_t out_row_stride, int out_dtype, void* stream) {
  if (!qweight || !scale || !out || N < 0 || K < 0 || q_row_stride < K) return IMQ_ERR_INVALID;
  hipStream_t st = (hipStream_t)stream;
  switch (s_dtype) {
    case IMQ_DT_BF16: return dequant8_out<IMQ_DT_BF16>(out_dtype, qweight, q_row_stride, scale, s_stride_n, N, K, out, out_row_stride, st);
    case IMQ_DT_FP16: return dequant8_out<IMQ_DT_FP16>(out_dtype, qweight, q_row_stride, scale, s_stride_n, N, K, out, out_row_stride, st);
    case IMQ_DT_FP32: return dequant8_out<IMQ_DT_FP32>(out_dtype, qweight, q_row_stride, scale, s_stride_n, N, K, out, out_row_stride, st);
  }
  return IMQ_ERR_INVALID;
}
