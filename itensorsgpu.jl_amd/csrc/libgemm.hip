// Plain FP64 GEMMs on the vendor library (rocBLAS). On large products its FP64
// MFMA kernels run at 61-76 TFLOP/s (4096^3, 8192x2048x10240,
// 10240x8192x2048) against 66 for the contraction kernel, whose point is the
// permutation fused into its loads: large contractions whose modes group into
// plain column-major matrices come here; the rest stay on the contraction
// kernel. Products inside a stream capture or a no-alloc call stay there too
// (the library may allocate its workspace).
#include <rocblas/rocblas.h>

#include <algorithm>
#include <climits>
#include <cstdlib>

#include "itg_internal.h"

namespace {

// products with a dimension below this stay on GETT: on the eigensolver's
// skinny back-transform products (32 to 128 rows or a K of 32 to 128) the
// library was slower (73.1 against 69.4 ms per n = 4096 eigendecomposition
// with them on it), and small products launch faster there
constexpr int64_t kLibMinDim = 256;
// and products with fewer multiply-adds than this, where the contraction
// kernel's choice of tile and K split is mostly the faster (us, library against
// it, NN / NT / TN): 256^3 18 18 18 / 8 8 9, 512 x 512 x 1000 35 34 35 / 22 20 24,
// 800^3 31 50 48 / 32 29 34, 2000 x 300 x 600 25 72 39 / 24 23 26; on the other
// side 2048 x 512 x 512 22 20 32 / 31 29 31, 1024^3 38 59 60 / 56 53 56,
// 1024 x 4096 x 512 66 65 64 / 74 75 74
constexpr double kLibMinWork = (double)(1 << 29);
// but for NN with 64 x 64 tiles for 0.75 of the CUs, or for 0.4 of them and K
// from 800 on, which the library runs at its full rate (us, library against
// native): 256 x 4096 x 300 14 / 20, 1500 x 600 x 500 22 / 30, 4200 x 400 x 300
// 27 / 30; 1379 x 344 x 802 (132 tiles) 21 / 26, 704 x 640 x 1100 (110) 26 / 31; on
// the other side 1079 x 666 x 491 (187 tiles) 21 / 21, 613 x 984 x 764 (160) 30 / 29,
// 1658 x 427 x 360 (182) 17 / 17, 344 x 1174 x 751 (114) 27 / 23, 679 x 372 x 1515
// (66) 34 / 31. NT and TN are split by the leading dimensions' alignment as much
// as by size, and stay with the rule above.
constexpr double kLibTilesNN = 0.75, kLibLongTilesNN = 0.4;
constexpr int64_t kLibLongNN = 800;
// The library does not split K: a product with tiles for less than this share
// of the CUs and a long K leaves most of the chip idle there, and the native
// kernel's K split is faster. us, library against native, NT: 1200 x 277 x 3878
// 123 / 70, 600 x 600 x 6000 182 / 105, 300 x 300 x 10000 274 to 1074 / 72,
// 700 x 277 x 1500 34 to 86 / 27; on the other side 512^3 12 / 18, 256 x 1280 x
// 512 19 / 21, 2000 x 400 x 5000 (224 tiles) 157 / 179. NN, which the library
// runs better: 354 x 1015 x 2681 (96 tiles) 57 / 50, 502 x 361 x 986 (48) 35 / 18;
// on the other side 822 x 497 x 1644 (104) 37 / 41, 712 x 639 x 1217 (120) 30 / 35,
// 341 x 1335 x 1291 (126) 31 / 38.
constexpr int64_t kLongK = 1024;
constexpr double kLongKTiles = 0.5, kLongKTilesNN = 0.4;

rocblas_handle handle_of(itg_ctx* ctx) {
  if (!ctx->blas) {
    rocblas_handle h = nullptr;
    if (rocblas_create_handle(&h) != rocblas_status_success) return nullptr;
    // no atomics: every call sums in a fixed order (bit-reproducible)
    rocblas_set_atomics_mode(h, rocblas_atomics_not_allowed);
    rocblas_set_pointer_mode(h, rocblas_pointer_mode_host);
    ctx->blas = h;
  }
  return (rocblas_handle)ctx->blas;
}

bool fits32(int64_t x) { return x >= 0 && x <= INT_MAX; }

rocblas_operation op_of(char t) {
  return (t == 'T' || t == 't') ? rocblas_operation_transpose : rocblas_operation_none;
}

}  // namespace

bool itg_libgemm_ok(itg_ctx* ctx, int dtype, int mode, char ta, char tb, int64_t m, int64_t n,
                    int64_t k) {
  if (!ctx->libgemm || dtype != ITG_F64 || mode != ITG_MODE_NATIVE) return false;
  if (ctx->fixed_ws) return false;
  if (!fits32(m) || !fits32(n) || !fits32(k)) return false;
  if (m < kLibMinDim || n < kLibMinDim || k < kLibMinDim) return false;
  const bool nn = (ta == 'N' || ta == 'n') && (tb == 'N' || tb == 'n');
  const double share = (double)((m + 63) / 64) * (double)((n + 63) / 64) / std::max(ctx->num_cu, 1);
  if (k >= kLongK && share < (nn ? kLongKTilesNN : kLongKTiles)) return false;
  if ((double)m * (double)n * (double)k < kLibMinWork &&
      !(nn && share >= (k >= kLibLongNN ? kLibLongTilesNN : kLibTilesNN)))
    return false;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &st) != hipSuccess) return false;
  return st == hipStreamCaptureStatusNone;
}

int itg_libgemm(itg_ctx* ctx, char ta, char tb, int64_t m, int64_t n, int64_t k, double alpha,
                const double* A, int64_t lda, const double* B, int64_t ldb, double beta,
                double* C, int64_t ldc) {
  if (!fits32(lda) || !fits32(ldb) || !fits32(ldc))
    return itg_fail(ctx, ITG_EUNSUPPORTED, "leading dimension beyond 32 bits");
  rocblas_handle h = handle_of(ctx);
  if (!h) return itg_fail(ctx, ITG_EHIP, "rocblas_create_handle failed");
  rocblas_set_stream(h, ctx->stream);
  const int t = itg_tstart(ctx, ITG_K_GETT);
  rocblas_status s = rocblas_dgemm(h, op_of(ta), op_of(tb), (rocblas_int)m, (rocblas_int)n,
                                   (rocblas_int)k, &alpha, A, (rocblas_int)lda, B,
                                   (rocblas_int)ldb, &beta, C, (rocblas_int)ldc);
  itg_tstop(ctx, t, ITG_K_GETT, 2.0 * m * n * k,
            8.0 * (m * k + k * n + m * n * (beta != 0.0 ? 2 : 1)));
  if (s != rocblas_status_success)
    return itg_fail(ctx, ITG_EHIP, "rocblas_dgemm: %s", rocblas_status_to_string(s));
  return ITG_OK;
}

void itg_libgemm_free(itg_ctx* ctx) {
  if (ctx->blas) {
    rocblas_destroy_handle((rocblas_handle)ctx->blas);
    ctx->blas = nullptr;
  }
}
