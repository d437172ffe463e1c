// Davidson eigensolver for one bond's two-site effective Hamiltonian, on the
// device: ITensors-style Krylov/Davidson (the eigsolve dmrg runs per bond,
// test/dmrg.jl:27) with the FP64 Krylov basis, Gram-Schmidt and Ritz
// combinations in fused passes on the device and the small projected
// eigenproblem on the host (cyclic Jacobi). In split-BF16
// mode the prepared Heff apply (five launches) is captured once into a HIP
// graph per (dims, basis slot) and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "itg_internal.h"

namespace {

constexpr int kMaxBasis = 17;   // maxiter + 1 <= 17

// The vector work of a step is a chain of passes over the basis, each needing
// the dot products of the one before. A pass leaves per-block partials, and
// every block of the next one sums them itself (in the same order, so all
// agree), so a Gram-Schmidt pass, its dot products and the norm never go
// through the host: per step eight launches and two read-backs (the projected
// matrix's new column and the residual norm) against 22 and five; a bond of
// 300 x 277, w = 14 with three Krylov vectors 0.87 -> 0.61 ms.
// Partials: nb x cnt, block b's k-th at part[b cnt + k].

// the cnt sums over nb blocks, in LDS (tot), for a 256-thread block
template <int MB>
__device__ __forceinline__ void block_totals(const double* __restrict__ part, int nb, int cnt,
                                             double (&sh)[4][MB], double (&tot)[MB]) {
  double s[MB];
#pragma unroll
  for (int k = 0; k < MB; ++k) s[k] = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256)
#pragma unroll
    for (int k = 0; k < MB; ++k)
      if (k < cnt) s[k] += part[(size_t)b * cnt + k];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < MB; ++k) {
    if (k >= cnt) break;
    double v = s[k];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) sh[w][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < cnt)
    tot[threadIdx.x] = (sh[0][threadIdx.x] + sh[1][threadIdx.x]) +
                       (sh[2][threadIdx.x] + sh[3][threadIdx.x]);
  __syncthreads();
}

// this block's cnt sums -> part
template <int MB>
__device__ __forceinline__ void write_partials(double (&s)[MB], int cnt, double (&sh)[4][MB],
                                               double* __restrict__ part) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < MB; ++k) {
    if (k >= cnt) break;
    double v = s[k];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) sh[w][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < cnt)
    part[(size_t)blockIdx.x * cnt + threadIdx.x] =
        (sh[0][threadIdx.x] + sh[1][threadIdx.x]) + (sh[2][threadIdx.x] + sh[3][threadIdx.x]);
}

// partials of V_k . x (V_k = V + k n), k < cnt
template <int MB>
__global__ __launch_bounds__(256) void dots_kernel(int64_t n, const double* __restrict__ V,
                                                   int cnt, const double* __restrict__ x,
                                                   double* __restrict__ part) {
  __shared__ double sh[4][MB];
  double s[MB];
#pragma unroll
  for (int k = 0; k < MB; ++k) s[k] = 0.0;
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    const double xi = x[i];
#pragma unroll
    for (int k = 0; k < MB; ++k)
      if (k < cnt) s[k] += V[(size_t)k * n + i] * xi;
  }
  write_partials<MB>(s, cnt, sh, part);
}

// y = x - sum_k h_k V_k, h the totals of `pin`; then partials of V_k . y
// (norm 0) or of y . y (norm 1)
template <int MB>
__global__ __launch_bounds__(256) void project_kernel(int64_t n, const double* __restrict__ V,
                                                      int cnt, const double* x, double* y,
                                                      const double* __restrict__ pin, int nb,
                                                      int norm, double* __restrict__ pout) {
  __shared__ double sh[4][MB], h[MB];
  block_totals<MB>(pin, nb, cnt, sh, h);
  double s[MB];
#pragma unroll
  for (int k = 0; k < MB; ++k) s[k] = 0.0;
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    double v[MB], yi = x[i];
#pragma unroll
    for (int k = 0; k < MB; ++k) {
      v[k] = k < cnt ? V[(size_t)k * n + i] : 0.0;
      if (k < cnt) yi -= h[k] * v[k];
    }
    y[i] = yi;
    if (norm) {
      s[0] += yi * yi;
    } else {
#pragma unroll
      for (int k = 0; k < MB; ++k) s[k] += v[k] * yi;
    }
  }
  __syncthreads();   // sh is reused
  write_partials<MB>(s, norm ? 1 : cnt, sh, pout);
}

// y = x / sqrt(total of pin); the total goes to *out
__global__ __launch_bounds__(256) void normalise_kernel(int64_t n, const double* x, double* y,
                                                        const double* __restrict__ pin, int nb,
                                                        double* out) {
  __shared__ double sh[4][1], h[1];
  block_totals<1>(pin, nb, 1, sh, h);
  const double f = 1.0 / sqrt(h[0]);
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) y[i] = f * x[i];
  if (blockIdx.x == 0 && threadIdx.x == 0 && out) *out = h[0];
}

struct Coefs {
  double c[kMaxBasis];
};

// phi = sum_k u_k V_k and, if q, q = sum_k u_k AV_k - lam phi; partials of
// (phi . phi, q . q)
template <int MB>
__global__ __launch_bounds__(256) void ritz_kernel(int64_t n, const double* __restrict__ V,
                                                   const double* __restrict__ AV, int cnt,
                                                   Coefs u, double lam, double* __restrict__ phi,
                                                   double* __restrict__ q,
                                                   double* __restrict__ part) {
  __shared__ double sh[4][2];
  double s[2] = {0.0, 0.0};
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    double p = 0.0, r = 0.0;
#pragma unroll
    for (int k = 0; k < MB; ++k)
      if (k < cnt) {
        p += u.c[k] * V[(size_t)k * n + i];
        if (q) r += u.c[k] * AV[(size_t)k * n + i];
      }
    phi[i] = p;
    s[0] += p * p;
    if (q) {
      r -= lam * p;
      q[i] = r;
      s[1] += r * r;
    }
  }
  write_partials<2>(s, 2, sh, part);
}

// q = a - lam v with lam the total of `pin` (also to out[0]); partials of q . q
__global__ __launch_bounds__(256) void residual_kernel(int64_t n, const double* __restrict__ a,
                                                       const double* __restrict__ v,
                                                       const double* __restrict__ pin, int nb,
                                                       double* __restrict__ q,
                                                       double* __restrict__ pout, double* out) {
  __shared__ double sh[4][1], h[1];
  block_totals<1>(pin, nb, 1, sh, h);
  double s[1] = {0.0};
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    const double r = a[i] - h[0] * v[i];
    q[i] = r;
    s[0] += r * r;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *out = h[0];
  __syncthreads();   // sh is reused
  write_partials<1>(s, 1, sh, pout);
}

__global__ __launch_bounds__(256) void totals_kernel(int nb, int cnt,
                                                     const double* __restrict__ part,
                                                     double* out) {
  __shared__ double sh[4][kMaxBasis], tot[kMaxBasis];
  block_totals<kMaxBasis>(part, nb, cnt, sh, tot);
  if (threadIdx.x < cnt) out[threadIdx.x] = tot[threadIdx.x];
}

// y = beta * y + alpha x
__global__ void axpby_kernel(int64_t n, double alpha, const double* __restrict__ x, double beta,
                             double* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = alpha * x[i] + (beta == 0.0 ? 0.0 : beta * y[i]);
}

// Launches of the passes on one context. Results for the host are written by
// the kernels into the context's pinned buffer: slots 0.. from totals, 20 and
// 21 from normalise and residual.
struct Passes {
  itg_ctx* ctx;
  int64_t n;
  static constexpr int kPart = 5000;   // doubles per partial buffer
  double* part(int i) const { return ctx->red + 32 + i * kPart; }
  double* host() const { return ctx->red_host; }
  // blocks of a pass with cnt sums: about 1024 elements each, at most 1024
  // (enough to stream from HBM) and at most the partial buffer's room
  int blocks(int cnt) const {
    const int64_t b = std::min<int64_t>({(n + 1023) / 1024, 1024, kPart / cnt});
    return (int)std::max<int64_t>(b, 1);
  }
  template <typename F>
  static void by_size(int cnt, F&& f) {   // f(integral constant >= cnt)
    if (cnt <= 2) f(std::integral_constant<int, 2>());
    else if (cnt <= 4) f(std::integral_constant<int, 4>());
    else if (cnt <= 8) f(std::integral_constant<int, 8>());
    else f(std::integral_constant<int, kMaxBasis>());
  }
  int dots(const double* V, int cnt, const double* x, int pout) const {
    by_size(cnt, [&](auto mb) {
      dots_kernel<mb()><<<blocks(cnt), 256, 0, ctx->stream>>>(n, V, cnt, x, part(pout));
    });
    ITG_LAUNCH_CHECK(ctx);
    return ITG_OK;
  }
  int project(const double* V, int cnt, const double* x, double* y, int pin, bool norm,
              int pout) const {
    by_size(cnt, [&](auto mb) {
      // the output partials hold cnt or one sum; one grid serves both
      project_kernel<mb()><<<blocks(cnt), 256, 0, ctx->stream>>>(n, V, cnt, x, y, part(pin),
                                                                 blocks(cnt), norm ? 1 : 0,
                                                                 part(pout));
    });
    ITG_LAUNCH_CHECK(ctx);
    return ITG_OK;
  }
  // nb: blocks that left the partials
  int normalise(const double* x, double* y, int pin, int nb) const {
    normalise_kernel<<<blocks(1), 256, 0, ctx->stream>>>(n, x, y, part(pin), nb, host() + 20);
    ITG_LAUNCH_CHECK(ctx);
    return ITG_OK;
  }
  int residual(const double* a, const double* v, int pin, double* q, int pout) const {
    residual_kernel<<<blocks(1), 256, 0, ctx->stream>>>(n, a, v, part(pin), blocks(1), q,
                                                        part(pout), host() + 21);
    ITG_LAUNCH_CHECK(ctx);
    return ITG_OK;
  }
  int ritz(const double* V, const double* AV, int cnt, const double* u, double lam, double* phi,
           double* q, int pout) const {
    Coefs c;
    for (int k = 0; k < kMaxBasis; ++k) c.c[k] = k < cnt ? u[k] : 0.0;
    by_size(cnt, [&](auto mb) {
      ritz_kernel<mb()><<<blocks(2), 256, 0, ctx->stream>>>(n, V, AV, cnt, c, lam, phi, q,
                                                            part(pout));
    });
    ITG_LAUNCH_CHECK(ctx);
    return ITG_OK;
  }
  // totals of cnt partials to the host's slots 0.., and wait
  int fetch(int pin, int cnt) const {
    totals_kernel<<<1, 256, 0, ctx->stream>>>(blocks(cnt), cnt, part(pin), host());
    ITG_LAUNCH_CHECK(ctx);
    ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return ITG_OK;
  }
};

// lowest eigenpair of the symmetric m x m matrix M (row-major) by cyclic
// Jacobi; u normalised with u[0] >= 0
void small_lowest(int m, const double* M, double* lam, double* u) {
  std::vector<double> a(M, M + m * m), v(m * m, 0.0);
  for (int i = 0; i < m; ++i) v[i * m + i] = 1.0;
  for (int sweep = 0; sweep < 100; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int i = 0; i < m; ++i)
      for (int j = 0; j < m; ++j) {
        tot += a[i * m + j] * a[i * m + j];
        if (i != j) off += a[i * m + j] * a[i * m + j];
      }
    if (off <= 1e-32 * tot || off == 0.0) break;
    for (int p = 0; p < m - 1; ++p)
      for (int q = p + 1; q < m; ++q) {
        double apq = a[p * m + q];
        if (apq == 0.0) continue;
        double theta = (a[q * m + q] - a[p * m + p]) / (2.0 * apq);
        double t = std::copysign(1.0, theta) / (std::fabs(theta) + std::sqrt(theta * theta + 1.0));
        double c = 1.0 / std::sqrt(t * t + 1.0), s = t * c;
        for (int k = 0; k < m; ++k) {
          double akp = a[k * m + p], akq = a[k * m + q];
          a[k * m + p] = c * akp - s * akq;
          a[k * m + q] = s * akp + c * akq;
        }
        for (int k = 0; k < m; ++k) {
          double apk = a[p * m + k], aqk = a[q * m + k];
          a[p * m + k] = c * apk - s * aqk;
          a[q * m + k] = s * apk + c * aqk;
        }
        for (int k = 0; k < m; ++k) {
          double vkp = v[k * m + p], vkq = v[k * m + q];
          v[k * m + p] = c * vkp - s * vkq;
          v[k * m + q] = s * vkp + c * vkq;
        }
      }
  }
  int best = 0;
  for (int i = 1; i < m; ++i)
    if (a[i * m + i] < a[best * m + best]) best = i;
  *lam = a[best * m + best];
  double nrm = 0.0;
  for (int k = 0; k < m; ++k) nrm += v[k * m + best] * v[k * m + best];
  nrm = std::sqrt(nrm);
  double sg = v[best] < 0.0 ? -1.0 : 1.0;
  for (int k = 0; k < m; ++k) u[k] = sg * v[k * m + best] / nrm;
}

// Heff apply x -> y, through a captured graph in split-BF16 mode
int heff_apply_graph(itg_ctx* ctx, int dtype, int mode, const int64_t* dims, const void* L,
                     const void* R, const void* prep, const void* x, void* y, void* work) {
  if (mode != ITG_MODE_BF16X3 || ctx->timing)
    return itg_heff2_apply_internal(ctx, dtype, mode, dims, L, R, prep, x, y, work);
  char key[256];
  std::snprintf(key, sizeof key, "%d/%d/%lld,%lld,%lld,%lld,%lld,%lld/%p/%p/%p/%p", dtype, mode,
                (long long)dims[0], (long long)dims[1], (long long)dims[2], (long long)dims[3],
                (long long)dims[4], (long long)dims[5], prep, x, y, work);
  auto it = ctx->graphs.find(key);
  if (it == ctx->graphs.end()) {
    // first use: eager (it also runs any one-time set-up outside a capture)
    ctx->graphs[key] = nullptr;
    return itg_heff2_apply_internal(ctx, dtype, mode, dims, L, R, prep, x, y, work);
  }
  if (!it->second) {
    if (ctx->graphs.size() > 256) {
      for (auto& kv : ctx->graphs)
        if (kv.second) hipGraphExecDestroy(kv.second);
      ctx->graphs.clear();
      return itg_heff2_apply_internal(ctx, dtype, mode, dims, L, R, prep, x, y, work);
    }
    hipGraph_t g = nullptr;
    ITG_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeRelaxed));
    int rc = itg_heff2_apply_internal(ctx, dtype, mode, dims, L, R, prep, x, y, work);
    hipError_t ce = hipStreamEndCapture(ctx->stream, &g);
    if (rc || ce != hipSuccess || !g) {
      if (g) hipGraphDestroy(g);
      hipGetLastError();
      return rc ? rc : itg_fail(ctx, ITG_EHIP, "heff graph capture failed");
    }
    hipGraphExec_t ge = nullptr;
    hipError_t ie = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (ie != hipSuccess) {
      hipGetLastError();
      return itg_fail(ctx, ITG_EHIP, "heff graph instantiate failed: %s", hipGetErrorString(ie));
    }
    it->second = ge;
  }
  ITG_HIP(ctx, hipGraphLaunch(it->second, ctx->stream));
  return ITG_OK;
}

}  // namespace

void itg_graph_cache_clear(itg_ctx* ctx) {
  for (auto& kv : ctx->graphs)
    if (kv.second) hipGraphExecDestroy(kv.second);
  ctx->graphs.clear();
}

extern "C" int64_t itg_davidson2_work_elems(int64_t chiL, int64_t d, int64_t chiR, int maxiter) {
  int64_t n = chiL * d * d * chiR;
  if (maxiter < 1) maxiter = 1;
  return (int64_t)(2 * (maxiter + 1) + 3) * n + 64;
}

// The learned Davidson preconditioner run inside the device loop: feature
// rows of the residual, the fused network, scatter, plus the skip step
// (0 none, 1 the residual, 2 the diagonal step), each skip at rms 1.
struct LearnedStep {
  const float* params = nullptr;
  int in = 0, hidden = 0, out = 0;
  int skip = 2;
  int net_steps = 0;        // Davidson steps per call that try the network (0: all)
  double floor = 1e-8;
  float* X = nullptr;       // rows x in
  float* Y = nullptr;       // rows x out
  float* work = nullptr;    // activations when the fused kernel does not fit
  double* tskip = nullptr;  // n doubles
};

static int learned_correction(itg_ctx* ctx, const LearnedStep& ls, int64_t chiL, int64_t d,
                              int64_t chiR, const double* q, const double* diag, double lam,
                              double* t) {
  const int64_t rows = chiL * chiR, n = rows * d * d;
  int rc = itg_mlp_features(ctx, chiL, d, chiR, q, diag, lam, ls.floor, 0, 1, rows, ls.X);
  if (rc) return rc;
  rc = itg_mlp_infer(ctx, (int)rows, ls.in, ls.hidden, ls.out, ls.params, ls.X, ls.Y, ls.work);
  if (rc) return rc;
  rc = itg_mlp_scatter(ctx, chiL, d, chiR, ls.Y, 0, rows, t);
  if (rc) return rc;
  if (ls.skip == 0) return ITG_OK;
  const double* sv = q;
  if (ls.skip == 2) {
    rc = itg_precond_diag(ctx, ITG_F64, n, q, diag, lam, ls.floor, ls.tskip);
    if (rc) return rc;
    sv = ls.tskip;
  }
  const Passes ps{ctx, n};
  rc = ps.dots(sv, 1, sv, 0);
  if (rc) return rc;
  rc = ps.fetch(0, 1);
  if (rc) return rc;
  const double sn = std::sqrt(ps.host()[0]);
  double sc = sn > 0.0 ? std::sqrt((double)n) / sn : 0.0;
  axpby_kernel<<<itg_blocks(n, 256, 8192), 256, 0, ctx->stream>>>(n, sc, sv, 1.0, t);
  ITG_LAUNCH_CHECK(ctx);
  return ITG_OK;
}

// ITensors' davidson on one bond with the basis on the device. With a
// learned step, each correction is first taken with the network and kept
// only if it lowers the residual norm; otherwise the basis vector is dropped,
// the previous Ritz pair restored and the diagonal step taken (`reverted`
// counts these).
static int davidson2_core(itg_ctx* ctx, int dtype, int mode, int64_t chiL, int64_t wl, int64_t wm,
                          int64_t wr, int64_t d, int64_t chiR, const void* L, const void* R,
                          const void* prep, void* psi, int maxiter, double errgoal,
                          const void* diag, const LearnedStep* ls, void* work, void* kwork,
                          double* energy, int* matvecs, int* reverted) {
  ITG_CHECK_CTX(ctx);
  if (dtype != ITG_F64) return itg_fail(ctx, ITG_EDTYPE, "davidson2: FP64 vectors only");
  if (maxiter < 1 || maxiter + 1 > kMaxBasis)
    return itg_fail(ctx, ITG_EARG, "davidson2: maxiter %d outside [1, %d]", maxiter,
                    kMaxBasis - 1);
  if (!psi || !prep || !work || !kwork || !energy)
    return itg_fail(ctx, ITG_EARG, "davidson2: null pointer");
  const int64_t dims[6] = {chiL, wl, wm, wr, d, chiR};
  const int64_t n = chiL * d * d * chiR;
  if (n <= 0) return itg_fail(ctx, ITG_EDIM, "davidson2: empty vector");
  if (maxiter > n - 1) maxiter = (int)std::max<int64_t>(n - 1, 0);
  const bool learned = ls != nullptr && ls->params != nullptr;
  double* V = (double*)kwork;                      // basis, maxiter + 1 vectors
  double* AV = V + (size_t)(maxiter + 1) * n;       // Heff applied to the basis
  double* q = AV + (size_t)(maxiter + 1) * n;       // residual
  double* t = q + n;                                // correction
  double* phi = t + n;                              // Ritz vector
  double u[kMaxBasis];
  int rc;
  const Passes ps{ctx, n};
  const double* h = ps.host();   // slots valid after a fetch
  // V0 = psi / |psi|, AV0, lam = V0 . AV0, q = AV0 - lam V0
  if ((rc = ps.dots((const double*)psi, 1, (const double*)psi, 0))) return rc;
  if ((rc = ps.normalise((const double*)psi, V, 0, ps.blocks(1)))) return rc;
  rc = heff_apply_graph(ctx, dtype, mode, dims, L, R, prep, V, AV, work);
  if (rc) return rc;
  if ((rc = ps.dots(V, 1, AV, 0))) return rc;
  if ((rc = ps.residual(AV, V, 0, q, 1))) return rc;
  if ((rc = ps.fetch(1, 1))) return rc;
  if (!(h[20] > 0.0)) return itg_fail(ctx, ITG_EARG, "davidson2: zero start vector");
  double lam = h[21], last = NAN, qn = std::sqrt(h[0]);
  int nmv = 1, m = 1, nrev = 0;
  std::vector<double> M(kMaxBasis * kMaxBasis, 0.0);
  M[0] = lam;
  u[0] = 1.0;
  for (int ni = 1; ni <= maxiter; ++ni) {
    bool conv = (qn < errgoal && std::fabs(lam - last) < errgoal) ||
                qn < std::max(1e-12, errgoal * 1e-3);
    if (qn < 1e-20 || (conv && ni > 1)) break;
    last = lam;
    bool stepped = false;
    const bool try_net = learned && (ls->net_steps <= 0 || ni <= ls->net_steps);
    const int attempts = try_net ? 2 : 1;
    for (int att = 0; att < attempts && !stepped; ++att) {
      const bool net = try_net && att == 0;
      const bool guarded = net;   // the diagonal step is the fallback
      // correction
      const double* t0 = t;
      rc = ITG_OK;
      if (net) rc = learned_correction(ctx, *ls, chiL, d, chiR, q, (const double*)diag, lam, t);
      else if (diag) rc = itg_precond_diag(ctx, ITG_F64, n, q, diag, lam, 1e-8, t);
      else t0 = q;
      if (rc) return rc;
      // two Gram-Schmidt passes against the basis, then V_m = t / |t|
      if ((rc = ps.dots(V, m, t0, 0))) return rc;
      if ((rc = ps.project(V, m, t0, t, 0, false, 1))) return rc;
      if ((rc = ps.project(V, m, t, t, 1, true, 2))) return rc;
      if ((rc = ps.normalise(t, V + (size_t)m * n, 2, ps.blocks(m)))) return rc;
      rc = heff_apply_graph(ctx, dtype, mode, dims, L, R, prep, V + (size_t)m * n,
                            AV + (size_t)m * n, work);
      if (rc) return rc;
      if ((rc = ps.dots(V, m + 1, AV + (size_t)m * n, 0))) return rc;
      if ((rc = ps.fetch(0, m + 1))) return rc;
      // a correction inside the basis: its product (in flight by now) is
      // dropped
      const double tn = std::sqrt(h[20]);
      if (tn < 1e-14 * std::max(1.0, qn)) {
        if (guarded) {
          ++nrev;
          continue;
        }
        break;
      }
      // the Ritz pair before this step, restored if the step is reverted
      const std::vector<double> Mprev(M.begin(), M.begin() + m * m);
      const double lamprev = lam;
      double uprev[kMaxBasis];
      for (int k = 0; k < m; ++k) uprev[k] = u[k];
      ++nmv;
      ++m;
      std::vector<double> Mn(m * m);
      for (int a = 0; a < m - 1; ++a)
        for (int b = 0; b < m - 1; ++b) Mn[a * m + b] = M[a * (m - 1) + b];
      for (int k = 0; k < m; ++k) Mn[k * m + (m - 1)] = Mn[(m - 1) * m + k] = h[k];
      M.assign(Mn.begin(), Mn.end());
      small_lowest(m, M.data(), &lam, u);
      // phi = sum u_k V_k, q = sum u_k AV_k - lam phi; nothing reads the
      // residual of the last step
      const bool lastq = ni == maxiter && !guarded;
      if ((rc = ps.ritz(V, AV, m, u, lam, phi, lastq ? nullptr : q, 0))) return rc;
      if (!lastq) {
        if ((rc = ps.fetch(0, 2))) return rc;
        const double qn_new = std::sqrt(h[1]);
        if (guarded && !(qn_new < qn)) {
          // the learned step did not lower the residual: drop it
          --m;
          M.assign(Mprev.begin(), Mprev.end());
          lam = lamprev;
          for (int k = 0; k < m; ++k) u[k] = uprev[k];
          if ((rc = ps.ritz(V, AV, m, u, lam, phi, q, 0))) return rc;
          ++nrev;
          continue;
        }
        qn = qn_new;
      }
      stepped = true;
    }
    if (!stepped) break;
  }
  // psi = Ritz vector (V0 when no step was taken), normalised
  const double* src = (m == 1) ? V : phi;
  if ((rc = ps.dots(src, 1, src, 0))) return rc;
  if ((rc = ps.normalise(src, (double*)psi, 0, ps.blocks(1)))) return rc;
  *energy = lam;
  if (matvecs) *matvecs = nmv;
  if (reverted) *reverted = nrev;
  return ITG_OK;
}

extern "C" int itg_davidson2(itg_ctx* ctx, int dtype, int mode, int64_t chiL, int64_t wl,
                             int64_t wm, int64_t wr, int64_t d, int64_t chiR, const void* L,
                             const void* R, const void* prep, void* psi, int maxiter,
                             double errgoal, const void* diag, void* work, void* kwork,
                             double* energy, int* matvecs) {
  return davidson2_core(ctx, dtype, mode, chiL, wl, wm, wr, d, chiR, L, R, prep, psi, maxiter,
                        errgoal, diag, nullptr, work, kwork, energy, matvecs, nullptr);
}

static bool mlp_fused(int in, int hidden, int out) {
  return hidden == 256 && ((in <= 16 && out <= 4) || (in <= 32 && out <= 9));
}

extern "C" int64_t itg_davidson2_mlp_work_elems(int64_t chiL, int64_t d, int64_t chiR,
                                                int hidden) {
  const int64_t rows = chiL * chiR, in = 3 * d * d, out = d * d;
  int64_t f = rows * in + rows * out + 2 * rows * d * d + 64;
  if (!mlp_fused((int)in, hidden, (int)out)) f += 2 * rows * (int64_t)hidden;
  return f;
}

extern "C" int itg_davidson2_mlp(itg_ctx* ctx, int dtype, int mode, int64_t chiL, int64_t wl,
                                 int64_t wm, int64_t wr, int64_t d, int64_t chiR, const void* L,
                                 const void* R, const void* prep, void* psi, int maxiter,
                                 double errgoal, const void* diag, const float* params,
                                 int hidden, int skip, int net_steps, double floor, void* mwork,
                                 void* work, void* kwork, double* energy, int* matvecs,
                                 int* reverted) {
  ITG_CHECK_CTX(ctx);
  if (!diag || !params || !mwork)
    return itg_fail(ctx, ITG_EARG, "davidson2_mlp: diagonal, parameters and work are required");
  if (skip < 0 || skip > 2) return itg_fail(ctx, ITG_EARG, "davidson2_mlp: skip %d", skip);
  if (!(floor > 0.0)) return itg_fail(ctx, ITG_EARG, "davidson2_mlp: floor must be > 0");
  const int64_t rows = chiL * chiR;
  if (rows <= 0 || rows > 0x7fffffff) return itg_fail(ctx, ITG_EDIM, "davidson2_mlp: rows");
  LearnedStep ls;
  ls.params = params;
  ls.in = (int)(3 * d * d);
  ls.hidden = hidden;
  ls.out = (int)(d * d);
  ls.skip = skip;
  ls.net_steps = net_steps;
  ls.floor = floor;
  // work: X | Y | tskip (n doubles, 8-byte aligned) | activations
  float* w = (float*)mwork;
  ls.X = w;
  ls.Y = ls.X + rows * ls.in;
  size_t off = (size_t)(rows * ls.in + rows * ls.out);
  off = (off + 1) & ~(size_t)1;
  ls.tskip = (double*)(w + off);
  off += 2 * (size_t)rows * d * d;
  ls.work = mlp_fused(ls.in, hidden, ls.out) ? nullptr : w + off;
  return davidson2_core(ctx, dtype, mode, chiL, wl, wm, wr, d, chiR, L, R, prep, psi, maxiter,
                        errgoal, diag, &ls, work, kwork, energy, matvecs, reverted);
}
