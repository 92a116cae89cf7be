// C-ABI entry points of the fused dequant linear family (imq_linear_w4 / _w2 / _w8) and the
// ABI metadata calls. Dispatch: decode rows (M <= 16) go to the MFMA decode kernels (gemv.hip; int8 from 5
// rows and int4 / int2 rows of no whole line-step to the short-batch forms, gemm_wk.hip), prefill rows to the
// GEMMs (gemm.hip); shapes or alignments a fast kernel rejects fall back to the
// generic dequantize-then-matmul kernel (never wrong, just slower).
//
// imq_linear_w4_noalloc is imq_linear_w4 with its workspace taken from a static per-device
// scratch array instead of a caller buffer (for callers that cannot allocate device memory).
#include <atomic>
#include <mutex>

#include "imq_common.h"

namespace imq {
int skinny_w4(const uint16_t* x, int64_t sxm, int64_t M, int64_t Kpad, const uint8_t* q, int64_t sqn,
              const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg,
              int zdt, int64_t N, int64_t G, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st,
              bool tiled);
int64_t ksplit_workspace_bytes(int64_t M, int64_t N, int64_t Kpad);
int64_t w4_decode_workspace_bytes(int64_t M, int64_t Kpad, int64_t G, int64_t N, int64_t sqn, int64_t sxm,
                                  int64_t ssn, int64_t ssg, int64_t szn, int64_t szg, int sdt, int zdt);
int skinny_w2(const uint16_t* x, int64_t sxm, int64_t M, int64_t Kpad, const uint8_t* q, int64_t sqn,
              const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg,
              int zdt, int64_t N, int64_t G, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st,
              bool tiled);
int64_t ksplit2_workspace_bytes(int64_t M, int64_t N, int64_t Kpad);
int skinny_w8(const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const int8_t* q, int64_t sqn,
              const void* sc, int64_t ssn, int sdt, int64_t N, uint16_t* y, int64_t sym, hipStream_t st,
              bool tiled);
int gemm_wq(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
            const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg,
            int zdt, int64_t N, int64_t G, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st);
int gemm_wq_tiled(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, const void* sc,
                  int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg, int zdt, int64_t N,
                  uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st);
int64_t gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, bool pair16);
int decode_plan_query(int kind, const int64_t* in, int64_t* out);
void gemm_plan_query(int64_t M, int64_t N, int64_t K, int cus, int64_t* out);
void wk_plan_query(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, int max_lds, int64_t* out);
void rbm_plan_query(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, int64_t* out);
void rb_plan_query(int bits, int64_t M, int64_t N, int64_t K, int64_t G, int cus, int64_t* out);
int gemm_wkd(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
             const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg, int zdt,
             int64_t N, int64_t G, uint16_t* y, int64_t sym, hipStream_t st);
// Whether decode rows go to the folded short-batch form before the skinny kernels: K not whole line-steps (no
// line or K-split kernel reads it), and
//   * many activations, as the skinny kernels' time steps up with what they stage: int4 from 72 K elements, where they
//     no longer fit the LDS and are staged in chunks, int2 from 33 K; or
//   * more than 8 rows of a longer K over at most one 32-column workgroup per CU (int4: over more than half the CUs;
//     below that its skinny kernel is not short of tiles either).
// us, cold weights, skinny -> folded: int4 6272 -> 9728 M = 10 / 12 21 / 41 -> 23.5 / 24, 11136 -> 5120 M = 6 / 7 29 / 41 -> 18 / 18,
// 2944 -> 5120 M = 8 / 9 / 16 9.3 / 9.7 / 11.4 -> 8.6 / 8.5 / 8.7, 2944 -> 2560 M = 9 / 16 6.8 / 9.0 -> 8.5 / 8.8, 2944 -> 9728 M = 9 /
// 16 12 / 14 -> 16 / 18; int2 3328 -> 9728 M = 9 / 12 15 / 20 -> 15 / 15, 11008 -> 5120 M = 8 / 16 43 / 65 -> 15 / 17, 2304 -> 1024
// M = 9 / 14 7.8 / 9.4 -> 7.6 / 7.6, 2304 -> 18944 M = 12 / 16 19 / 26 -> 20 / 20.
bool folded_first(int bits, int64_t M, int64_t N, int64_t K) {
  if (M <= 4 || M > 16 || K % (1024 / bits) == 0) return false;
  if (M * K >= (bits == 4 ? 72 << 10 : 33 << 10)) return true;
  const int64_t tiles = imq_cdiv(N, 32), cus = device_info().cus;
  return M > 8 && K >= 2048 && tiles <= cus && (bits == 2 || 2 * tiles > cus);
}
// Whether the generic kernel (one wave per row) is the faster for rows no decode kernel takes: few rows of a short K,
// less than the folded form's staging and sum over 16 waves. us, generic against folded: 64 -> 1024 M = 1 / 16 3.9 / 5.3
// against 6.7 / 7.0, 128 -> 1024 M = 8 / 16 5.8 / 7.2 against 6.9 / 7.0, 320 -> 1024 M = 1 / 4 5.4 / 6.8 against 6.2 / 6.3,
// 64 -> 4096 M = 1 6.7 against 6.2.
bool generic_first(int64_t M, int64_t N, int64_t K) { return N <= 2048 && K * (M + 4) <= 2048; }
int gemm_wk(int bits, const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
            const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn, int64_t szg, int zdt,
            int64_t N, int64_t G, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st, bool tiled);
template <int BITS>
int generic_gemv(const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const uint8_t* q, int64_t sqn,
                 const void* sc, int64_t ssn, int64_t ssg, int sdt, const void* zr, int64_t szn,
                 int64_t szg, int zdt, int64_t N, int64_t G, uint16_t* y, int64_t sym, hipStream_t st);
}  // namespace imq

namespace {

bool dt_ok(int d) { return d == IMQ_DT_BF16 || d == IMQ_DT_FP16 || d == IMQ_DT_FP32; }

// Shared argument validation of the group-wise formats (int4 / int2).
int check_g(int bits, const void* x, int64_t sxm, int64_t M, int64_t Kpad, const void* q, int64_t sqn,
            const void* sc, int sdt, const void* zr, int zdt, int64_t N, int64_t G, const void* y,
            int64_t sym) {
  if (!x || !q || !sc || !zr || !y) return IMQ_ERR_INVALID;
  if (M < 0 || N < 0 || Kpad <= 0 || G <= 0 || Kpad % G != 0) return IMQ_ERR_INVALID;
  if ((Kpad * bits) % 8 != 0 || sqn < Kpad * bits / 8) return IMQ_ERR_INVALID;
  if (sxm < Kpad || sym < N) return IMQ_ERR_INVALID;
  if (!dt_ok(sdt) || !dt_ok(zdt)) return IMQ_ERR_INVALID;
  return IMQ_OK;
}

}  // namespace

extern "C" int imq_abi_version(void) { return IMQ_ABI_VERSION; }

extern "C" int64_t imq_linear_workspace_bytes(int64_t M, int64_t N, int64_t K_pad) {
  if (M < 0 || N < 0 || K_pad <= 0) return -1;
  const int64_t g = imq::gemm_workspace_bytes(M, N, K_pad, false);
  const int64_t d = imq::ksplit_workspace_bytes(M, N, K_pad);
  const int64_t d2 = imq::ksplit2_workspace_bytes(M, N, K_pad);
  const int64_t gd = g > d ? g : d;
  return gd > d2 ? gd : d2;
}

extern "C" int64_t imq_linear_w4_workspace_bytes(int64_t M, int64_t K_pad, int64_t N, int64_t group_size,
                                                 int64_t q_row_stride, int64_t x_row_stride, int64_t s_stride_n,
                                                 int64_t s_stride_g, int s_dtype, int64_t z_stride_n,
                                                 int64_t z_stride_g, int z_dtype) {
  if (M < 0 || N < 0 || K_pad <= 0 || group_size <= 0 || K_pad % group_size) return -1;
  if (M == 0 || N == 0) return 0;
  if (M > 16) return imq::gemm_workspace_bytes(M, N, K_pad, s_dtype == z_dtype && s_dtype != IMQ_DT_FP32);
  return imq::w4_decode_workspace_bytes(M, K_pad, group_size, N, q_row_stride, x_row_stride, s_stride_n, s_stride_g,
                                        z_stride_n, z_stride_g, s_dtype, z_dtype);
}

extern "C" int imq_launch_plan(int kind, const int64_t* in, int64_t* out) {
  if (!in || !out) return IMQ_ERR_INVALID;
  for (int i = 0; i < 5; ++i) out[i] = 0;
  const int64_t M = in[0], K = in[1], G = in[2], N = in[3];
  const int cus = (int)in[9];
  if (kind == IMQ_PLAN_GEMM) {
    if (M <= 16 || N <= 0 || K <= 0 || K % 64 != 0 || cus <= 0) return IMQ_OK;
    imq::gemm_plan_query(M, N, K, cus, out);
    return IMQ_OK;
  }
  if (kind == IMQ_PLAN_GEMM_RB) {
    if (cus <= 0) return IMQ_OK;
    imq::rb_plan_query(G == 0 ? 8 : 4, M, N, K, G == 0 ? 128 : G, cus, out);
    return IMQ_OK;
  }
  if (kind == IMQ_PLAN_GEMM_WK || kind == IMQ_PLAN_GEMM_RBM) {
    const int64_t bits = K > 0 ? in[4] * 8 / K : 0;
    if (cus <= 0 || N <= 0 || K <= 0 || (bits != 2 && bits != 4 && bits != 8)) return IMQ_OK;
    if (kind == IMQ_PLAN_GEMM_RBM) {
      imq::rbm_plan_query((int)bits, M, N, K, G, cus, out);
      return IMQ_OK;
    }
    imq::wk_plan_query((int)bits, M, N, K, G, cus, (int)in[8], out);
    return IMQ_OK;
  }
  if (in[7] != IMQ_DT_BF16 && in[7] != IMQ_DT_FP16 && in[7] != IMQ_DT_FP32) return IMQ_ERR_INVALID;
  return imq::decode_plan_query(kind, in, out);
}

extern "C" const char* imq_strerror(int status) {
  switch (status) {
    case IMQ_OK: return "ok";
    case IMQ_ERR_INVALID: return "invalid argument (shape, stride, dtype or null pointer)";
    case IMQ_ERR_UNSUPPORTED: return "configuration not supported by this kernel family";
    case IMQ_ERR_ALIGN: return "pointer or stride misaligned for this kernel";
    case IMQ_ERR_SCRATCH:
      return "workspace need exceeds the static scratch of the allocation-free entry point "
             "(IMQ_NOALLOC_SCRATCH_BYTES)";
  }
  if (status > 0) return hipGetErrorString((hipError_t)status);
  return "unknown status";
}

extern "C" int imq_linear_w4(const void* x, int64_t x_row_stride, int64_t M, int64_t K_pad,
                             const void* qweight, int64_t q_row_stride, const void* scale,
                             int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                             int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                             int64_t group_size, void* y, int64_t y_row_stride, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  int rc = check_g(4, x, x_row_stride, M, K_pad, qweight, q_row_stride, scale, s_dtype, zero, z_dtype, N,
                   group_size, y, y_row_stride);
  if (rc != IMQ_OK) return rc;
  if (M == 0 || N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* xb = (const uint16_t*)x;
  uint16_t* yb = (uint16_t*)y;
  const uint8_t* q = (const uint8_t*)qweight;
  if (imq::folded_first(4, M, N, K_pad)) {
    rc = imq::gemm_wkd(4, xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype, zero,
                       z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, st);
    if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  }
  if (M <= 16) {
    rc = imq::skinny_w4(xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype,
                        zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, workspace,
                        workspace_bytes, st, false);
  } else {
    rc = imq::gemm_wq(4, xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g,
                      s_dtype, zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride,
                      workspace, workspace_bytes, st);
  }
  if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  if (!imq::generic_first(M, N, K_pad)) {
    rc = imq::gemm_wkd(4, xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype, zero,
                       z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, st);
    if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  }
  return imq::generic_gemv<4>(xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g,
                              s_dtype, zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb,
                              y_row_stride, st);
}

// int4 weights in the line-tiled layout: the arguments and results of imq_linear_w4. The layout
// permutes 16-byte pieces within each 16-row tile (N a multiple of 16, dense rows of K_pad / 2
// bytes, K_pad a multiple of 256, groups of 128); the kernels that read it are the decode line,
// wave-split and K-split kernels and the prefill GEMMs. A call none of them takes (past 16 rows also one whose scale
// and zero differ in dtype) returns IMQ_ERR_UNSUPPORTED: no row-layout kernel may read these bytes.
extern "C" int imq_linear_w4_tiled(const void* x, int64_t x_row_stride, int64_t M, int64_t K_pad,
                                   const void* qweight, int64_t q_row_stride, const void* scale,
                                   int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                                   int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                                   int64_t group_size, void* y, int64_t y_row_stride, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  int rc = check_g(4, x, x_row_stride, M, K_pad, qweight, q_row_stride, scale, s_dtype, zero, z_dtype, N,
                   group_size, y, y_row_stride);
  if (rc != IMQ_OK) return rc;
  if (N % 16 != 0 || K_pad % 256 != 0 || group_size != 128 || q_row_stride != K_pad / 2) return IMQ_ERR_INVALID;
  if (M == 0 || N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* xb = (const uint16_t*)x;
  uint16_t* yb = (uint16_t*)y;
  const uint8_t* q = (const uint8_t*)qweight;
  if (M <= 16)
    return imq::skinny_w4(xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype,
                          zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, workspace,
                          workspace_bytes, st, true);
  return imq::gemm_wq_tiled(4, xb, x_row_stride, M, K_pad, q, scale, s_stride_n, s_stride_g, s_dtype, zero,
                            z_stride_n, z_stride_g, z_dtype, N, yb, y_row_stride, workspace, workspace_bytes, st);
}

// int2 weights in the line-tiled layout: the arguments and results of imq_linear_w2 (N a multiple of
// 16, dense rows of K_pad / 4 bytes, K_pad a multiple of 512, groups of 64); the decode line and
// K-split kernels and the prefill GEMMs read it, other calls return IMQ_ERR_UNSUPPORTED.
extern "C" int imq_linear_w2_tiled(const void* x, int64_t x_row_stride, int64_t M, int64_t K_pad,
                                   const void* qweight, int64_t q_row_stride, const void* scale,
                                   int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                                   int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                                   int64_t group_size, void* y, int64_t y_row_stride, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  int rc = check_g(2, x, x_row_stride, M, K_pad, qweight, q_row_stride, scale, s_dtype, zero, z_dtype, N,
                   group_size, y, y_row_stride);
  if (rc != IMQ_OK) return rc;
  if (N % 16 != 0 || K_pad % 512 != 0 || group_size != 64 || q_row_stride != K_pad / 4) return IMQ_ERR_INVALID;
  if (M == 0 || N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* xb = (const uint16_t*)x;
  uint16_t* yb = (uint16_t*)y;
  const uint8_t* q = (const uint8_t*)qweight;
  if (M <= 16)
    return imq::skinny_w2(xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype,
                          zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, workspace,
                          workspace_bytes, st, true);
  return imq::gemm_wq_tiled(2, xb, x_row_stride, M, K_pad, q, scale, s_stride_n, s_stride_g, s_dtype, zero,
                            z_stride_n, z_stride_g, z_dtype, N, yb, y_row_stride, workspace, workspace_bytes, st);
}

namespace {

// int8 decode rows: from 5 the short-batch GEMM where it takes them (wk_rows, gemm_wk.hip), else the
// line and skinny kernels. Of the workspace at most imq_linear_workspace_bytes is used, so a larger buffer
// kept for other calls changes no result.
int decode_w8(const uint16_t* x, int64_t sxm, int64_t M, int64_t K, const void* q, int64_t sqn, const void* sc, int64_t ssn,
              int sdt, int64_t N, uint16_t* y, int64_t sym, void* ws, int64_t wsb, hipStream_t st, bool tiled) {
  if (M > 4) {
    const int64_t own = imq_linear_workspace_bytes(M, N, K);
    const int rc = imq::gemm_wk(8, x, sxm, M, K, (const uint8_t*)q, sqn, sc, ssn, 0, sdt, nullptr, 0, 0, sdt, N, 0, y,
                                sym, ws, wsb < own ? wsb : own, st, tiled);
    if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  }
  return imq::skinny_w8(x, sxm, M, K, (const int8_t*)q, sqn, sc, ssn, sdt, N, y, sym, st, tiled);
}

}  // namespace

// int8 weights in the line-tiled layout: the arguments and results of imq_linear_w8 (N a multiple of
// 16, dense rows of K bytes, K a multiple of 128); the decode line and skinny kernels and both
// prefill GEMMs read it, other calls return IMQ_ERR_UNSUPPORTED.
extern "C" int imq_linear_w8_tiled(const void* x, int64_t x_row_stride, int64_t M, int64_t K,
                                   const void* qweight, int64_t q_row_stride, const void* scale,
                                   int64_t s_stride_n, int s_dtype, int64_t N, void* y, int64_t y_row_stride,
                                   void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x || !qweight || !scale || !y || M < 0 || N < 0 || K <= 0) return IMQ_ERR_INVALID;
  if (q_row_stride < K || x_row_stride < K || y_row_stride < N || !dt_ok(s_dtype)) return IMQ_ERR_INVALID;
  if (N % 16 != 0 || K % 128 != 0 || q_row_stride != K) return IMQ_ERR_INVALID;
  if (M == 0 || N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* xb = (const uint16_t*)x;
  uint16_t* yb = (uint16_t*)y;
  if (M <= 16)
    return decode_w8(xb, x_row_stride, M, K, qweight, q_row_stride, scale, s_stride_n, s_dtype, N, yb, y_row_stride,
                     workspace, workspace_bytes, st, true);
  return imq::gemm_wq_tiled(8, xb, x_row_stride, M, K, (const uint8_t*)qweight, scale, s_stride_n, 0, s_dtype,
                            nullptr, 0, 0, s_dtype, N, yb, y_row_stride, workspace, workspace_bytes, st);
}

// ---- allocation-free variant of imq_linear_w4 ----------------------------------------------------
// The scratch array: each device the library runs on holds its own copy until the process ends.
// Host code never uses the name `scratch` as an address (on the host it is only a stand-in for
// the symbol): the device address comes from hipGetSymbolAddress, once per device, and only that
// pointer is passed to kernels.
static __device__ __align__(256) unsigned char scratch[IMQ_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of the current device's scratch array, resolved on the first call per device
// (with that device current) and cached.
int scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return IMQ_ERR_UNSUPPORTED;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return (int)e;
      if (!p) return IMQ_ERR_UNSUPPORTED;
      g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return IMQ_OK;
}

}  // namespace

extern "C" int imq_linear_w4_noalloc(const void* x, int64_t x_row_stride, int64_t M, int64_t K_pad,
                                     const void* qweight, int64_t q_row_stride, const void* scale,
                                     int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                                     int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                                     int64_t group_size, void* y, int64_t y_row_stride, void* stream) {
  int rc = check_g(4, x, x_row_stride, M, K_pad, qweight, q_row_stride, scale, s_dtype, zero, z_dtype, N,
                   group_size, y, y_row_stride);
  if (rc != IMQ_OK) return rc;
  if (M == 0 || N == 0) return IMQ_OK;
  // The partials of the K-split / split-K launches need no initialisation (every element a
  // reduction reads is written first by the same call), so the array is never cleared. The need
  // is this call's own (the dispatcher's plans for these strides on this device): shapes whose
  // kernels keep their partials in the workgroup need none, whatever their size.
  const int64_t need = imq_linear_w4_workspace_bytes(M, K_pad, N, group_size, q_row_stride, x_row_stride, s_stride_n,
                                                     s_stride_g, s_dtype, z_stride_n, z_stride_g, z_dtype);
  if (need > IMQ_NOALLOC_SCRATCH_BYTES) return IMQ_ERR_SCRATCH;
  void* ws = nullptr;
  rc = scratch_ptr(&ws);
  if (rc != IMQ_OK) return rc;
  return imq_linear_w4(x, x_row_stride, M, K_pad, qweight, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype,
                       zero, z_stride_n, z_stride_g, z_dtype, N, group_size, y, y_row_stride, ws,
                       IMQ_NOALLOC_SCRATCH_BYTES, stream);
}

extern "C" int imq_linear_w2(const void* x, int64_t x_row_stride, int64_t M, int64_t K_pad,
                             const void* qweight, int64_t q_row_stride, const void* scale,
                             int64_t s_stride_n, int64_t s_stride_g, int s_dtype, const void* zero,
                             int64_t z_stride_n, int64_t z_stride_g, int z_dtype, int64_t N,
                             int64_t group_size, void* y, int64_t y_row_stride, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  int rc = check_g(2, x, x_row_stride, M, K_pad, qweight, q_row_stride, scale, s_dtype, zero, z_dtype, N,
                   group_size, y, y_row_stride);
  if (rc != IMQ_OK) return rc;
  if (M == 0 || N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* xb = (const uint16_t*)x;
  uint16_t* yb = (uint16_t*)y;
  const uint8_t* q = (const uint8_t*)qweight;
  if (imq::folded_first(2, M, N, K_pad)) {
    rc = imq::gemm_wkd(2, xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype, zero,
                       z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, st);
    if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  }
  if (M <= 16) {
    rc = imq::skinny_w2(xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype,
                        zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, workspace,
                        workspace_bytes, st, false);
  } else {
    rc = imq::gemm_wq(2, xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g,
                      s_dtype, zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride,
                      workspace, workspace_bytes, st);
  }
  if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  if (!imq::generic_first(M, N, K_pad)) {
    rc = imq::gemm_wkd(2, xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g, s_dtype, zero,
                       z_stride_n, z_stride_g, z_dtype, N, group_size, yb, y_row_stride, st);
    if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  }
  return imq::generic_gemv<2>(xb, x_row_stride, M, K_pad, q, q_row_stride, scale, s_stride_n, s_stride_g,
                              s_dtype, zero, z_stride_n, z_stride_g, z_dtype, N, group_size, yb,
                              y_row_stride, st);
}

extern "C" int imq_linear_w8(const void* x, int64_t x_row_stride, int64_t M, int64_t K,
                             const void* qweight, int64_t q_row_stride, const void* scale,
                             int64_t s_stride_n, int s_dtype, int64_t N, void* y, int64_t y_row_stride,
                             void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x || !qweight || !scale || !y || M < 0 || N < 0 || K <= 0) return IMQ_ERR_INVALID;
  if (q_row_stride < K || x_row_stride < K || y_row_stride < N || !dt_ok(s_dtype)) return IMQ_ERR_INVALID;
  if (M == 0 || N == 0) return IMQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* xb = (const uint16_t*)x;
  uint16_t* yb = (uint16_t*)y;
  int rc;
  if (M <= 16) {
    rc = decode_w8(xb, x_row_stride, M, K, qweight, q_row_stride, scale, s_stride_n, s_dtype, N, yb, y_row_stride,
                   workspace, workspace_bytes, st, false);
  } else {
    rc = imq::gemm_wq(8, xb, x_row_stride, M, K, (const uint8_t*)qweight, q_row_stride, scale, s_stride_n,
                      0, s_dtype, nullptr, 0, 0, s_dtype, N, 0, yb, y_row_stride, workspace, workspace_bytes, st);
  }
  if (rc != IMQ_ERR_UNSUPPORTED) return rc;
  return imq::generic_gemv<8>(xb, x_row_stride, M, K, (const uint8_t*)qweight, q_row_stride, scale,
                              s_stride_n, 0, s_dtype, nullptr, 0, 0, s_dtype, N, 1, yb, y_row_stride, st);
}
