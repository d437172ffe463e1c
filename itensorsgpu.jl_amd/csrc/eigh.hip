// Symmetric eigendecomposition with truncation, FP64 throughout: the
// `eigen(Hermitian)` step of factorize (src/tensor/culinearalgebra.jl:74-108:
// syevd, eigenvalues reversed to descending, truncate!, columns reversed and
// sliced) used by replacebond! on the density matrix rho = phi phi^T.
//
// 1. Householder tridiagonalisation. More than 3584 trailing rows: blocked as
//    in LAPACK dsytrd/dlatrd (panels of NB columns), per column two kernels
//    spanning the GPU (the reflector fused into the symmetric matrix-vector
//    product over the trailing block, then w and the next column's update; see
//    below), per panel the rank-2*NB trailing update A -= V W^T + W V^T on FP64
//    MFMA. Then in the registers of many workgroups that exchange one vector
//    pair per column, and the last 192 rows in one workgroup.
// 2. Divide and conquer on the tridiagonal (Cuppen tearing at every split,
//    bottom-up merges): blocks up to 64 in one launch; per larger merge a sort
//    + deflation workgroup, rotation, secular-root, Gu-Eisenstat and
//    eigenvector kernels, and Q_new = Q_old[:, nondeflated] V on MFMA (gathered
//    columns through a device offset table) for large merges.
// 3. Eigenvalues sorted descending, truncate! decided on the device, and only
//    the k kept eigenvectors back-transformed by the compact-WY block
//    reflectors (Schreiber & Van Loan 1989) on MFMA.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "dc_core.h"
#include "eigh2.h"
#include "gett.h"
#include "itg_internal.h"
#include "truncate_core.h"

int itg_truncate_device_async(itg_ctx* ctx, const double* P, int64_t n, int64_t maxdim,
                              int64_t mindim, double cutoff, int abs_cut, int rel_cut,
                              int semantics, double* out3);

namespace {

constexpr int NB = 32;          // tridiagonalisation panel width
constexpr int TWO_STAGE_MIN = 256;   // n from which the two-stage reduction runs
constexpr int SMALL_MERGE = 256;

__device__ double block_sum(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  int nw = (blockDim.x + 63) >> 6;
  for (int i = 0; i < nw; ++i) r += sh[i];
  return r;
}

// ------------------------------------------------------ lane exchanges
// On the vector unit (DPP within a row of 16 lanes, permlane swaps between
// rows): __shfl_xor goes through the LDS pipe, which the CU's waves share.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// lanes with bit MASK (32 or 16) clear: a summed over the pair of lanes that
// differ in it; the others: b
template <int MASK>
__device__ __forceinline__ double swap_add(double a, double b) {
  if constexpr (MASK == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  }
}

// the value of a lane that differs in bit MASK (8, 4, 2 or 1): for 8 and 4 its
// mirror image in the row or half row, which differs in the lower bits too
template <int MASK>
__device__ __forceinline__ double row_partner(double v) {
  if constexpr (MASK == 8) return dpp_d<0x140>(v);
  else if constexpr (MASK == 4) return dpp_d<0x141>(v);
  else if constexpr (MASK == 2) return dpp_d<0x4E>(v);
  else return dpp_d<0xB1>(v);
}

// sum over each row of 16 lanes, the same bits in all of them
__device__ __forceinline__ double row16_sum(double v) {
  v += row_partner<1>(v);
  v += row_partner<2>(v);
  v += row_partner<4>(v);
  v += row_partner<8>(v);
  return v;
}

// N values per lane -> d[0]: value number lane >> (6 - log2 N) summed over the
// lanes that differ in the bits used (64 / N lanes are left for each); every
// step halves the values a lane carries. MASK = 32 to begin with.
template <int N, int MASK, int M>
__device__ __forceinline__ void fold_halves(double (&d)[M], int lane) {
  if constexpr (N > 1) {
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      if constexpr (MASK >= 16) {
        d[k] = swap_add<MASK>(d[k], d[k + N / 2]);
      } else {
        const bool up = (lane & MASK) != 0;
        const double send = up ? d[k] : d[k + N / 2], keep = up ? d[k + N / 2] : d[k];
        d[k] = keep + row_partner<MASK>(send);
      }
    }
    fold_halves<N / 2, MASK / 2>(d, lane);
  }
}

// sum of v over the lanes that differ only in bits MASK, MASK / 2, ..., 1
template <int MASK>
__device__ __forceinline__ double fold_sum(double v) {
  if constexpr (MASK >= 16) v = swap_add<MASK>(v, v);
  else if constexpr (MASK >= 1) v += row_partner<MASK>(v);
  if constexpr (MASK > 1) return fold_sum<MASK / 2>(v);
  else return v;
}

// ------------------------------------------------------- tridiagonalisation
// Per column j (panel column i) two kernels run across the whole GPU:
//  trd_symv: one block per 64 x 64 tile on or below the diagonal of A22
//    leaves row and column partials of A22 a (a = column j below the
//    diagonal, one writer per slot) and a partial of a^T A22 a; these need
//    neither the reflector's norm nor its scale. Extra blocks form the
//    reflector from the norm partials left by the previous kernel and the
//    panel dots a = W^T v and b = V^T v; the grid stores v into the panel.
//  trd_post: y = A22 v = s (A22 a - beta A22(:, 0)), then
//    w = tau (y - V a - W b) + alpha v, where
//    alpha = -tau/2 w^T v = -tau^2/2 (y^T v - 2 a^T b) needs no extra
//    reduction pass; v goes into A; then the next panel column's update
//    A(:,j+1) -= V W(j+1,:)^T + W V(j+1,:)^T and the partial sums of its
//    squared tail for the next reflector.
constexpr int TRD_ROWS = 64;   // rows per block of the row-parallel kernels

// sum over the wave, the same bits in every lane
__device__ __forceinline__ double wave_sum(double v) { return fold_sum<32>(v); }

// sum over a 256-thread block, the same value returned to every thread and
// computed in the same order in every block (bitwise identical results)
__device__ __forceinline__ double block_sum256(double v, double* sh4) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh4[threadIdx.x >> 6] = v;
  __syncthreads();
  return (sh4[0] + sh4[1]) + (sh4[2] + sh4[3]);
}

__device__ __forceinline__ double sum_partials(const double* __restrict__ p, int np, double* sh4) {
  double s = 0.0;
  for (int b = threadIdx.x; b < np; b += 256) s += p[b];
  return block_sum256(s, sh4);
}

// partial sums of A[r, j]^2, r >= j+2, one per TRD_ROWS-row block
__global__ __launch_bounds__(256) void trd_colnorm_kernel(const double* __restrict__ A, int n, int j,
                                                          double* __restrict__ pnorm) {
  __shared__ double sh4[4];
  int r = blockIdx.x * TRD_ROWS + threadIdx.x;
  double s = 0.0;
  if (threadIdx.x < TRD_ROWS && r < n && r >= j + 2) {
    double a = A[r + (size_t)j * n];
    s = a * a;
  }
  s = block_sum256(s, sh4);
  if (threadIdx.x == 0) pnorm[blockIdx.x] = s;
}

// Symmetric product of the trailing matrix A22 (rows/cols o = j+1 .. n-1,
// local index l = r - o, size m) with column j itself, a(l) = A[o + l, j],
// reading only the 64 x 64 tiles on and below the diagonal (both triangles
// of a diagonal tile are stored, so it is used whole). The reflector is
// v = s (a - beta e0), s = 1 / (alpha - beta), so
//   A22 v = s (A22 a - beta A22(:, 0)),
//   v^T A22 v = s^2 (a^T A22 a - 2 beta (A22 a)(0) + beta^2 A22(0, 0)),
// and the tiles need neither the norm nor beta: the post kernel applies s
// and beta. Tile (I, J), I >= J, writes its row partial
// sum_{c in J} A[r,c] a[c] to Ypart[J][r] and, below the diagonal, its
// column partial sum_{r in I} A[r,c] a[r] to Ypart[I][c]: every (t, l) of
// Ypart (t < T tile rows) has exactly one writer and (A22 a)(l) =
// sum_t Ypart[t][l]. Its share of a^T A22 a goes to pyv[tile].
//
// Thread (wave w, lane l) keeps A[r0 + l, c0 + w + 4q], q < 16, in
// registers. Row partials are 16 products per thread summed over the four
// waves in LDS; column partials are sums over the 64 lanes, done for all 16
// columns of a wave at once by a transposing butterfly (each exchange halves
// the values a lane carries), after which lanes with l % 4 == 0 hold column
// w + 4 q(l), q(l) = 8 b5 + 4 b4 + 2 b3 + b2 from the lane's bits. With no
// tile in LDS eight blocks fit on a CU, so a 4096-row trailing block (2080
// tiles) is read in one round.
//
// Bound by that read: 67 MB against 32 MB of L2 (past it 6 TB/s, within it 14).
// A tile keeps its XCD from column to column (the dot blocks are padded to
// eight), and every other column walks the tiles backwards, so that the ones
// read last are still in L2: n = 4096 whole 43.0 -> 40.8 ms, 6000 109 -> 104.
//
// The first i blocks form the panel dots W(:,q).v and V(:,q).v, q < i; they,
// and the blocks that write v into the panel (and its mirror V2), form the
// reflector from the norm partials (identically in every block). Block 0
// stores d, e, tau and sc = {s, A22(0, 0)}.
constexpr int TS = 64;

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void trd_symv_kernel(
    const double* __restrict__ A, int n, int j, int i, const double* __restrict__ pnorm, int npn,
    double* __restrict__ Vp, const double* __restrict__ Wp, double* __restrict__ V2,
    double* __restrict__ Ypart, double* __restrict__ ab, double* __restrict__ pyv, int ntiles,
    double* d, double* e, double* tau, double* __restrict__ sc) {
  __shared__ double vr[TS], vc[TS];
  __shared__ double red[4][TS];
  __shared__ double sh4[4];
  const size_t ld = (size_t)n;
  const double* a = A + (size_t)j * ld;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int m = n - j - 1, o = j + 1;
  // the panel-dot blocks come first: each walks a whole column, so they
  // start before the tiles fill the machine
  const int nd = (i + 7) & ~7, b8 = (int)blockIdx.x - nd;
  int bid = b8;   // tile index, negative for the dots
  if (b8 >= 0 && (j & 1)) bid = (((ntiles + 7) >> 3) - 1 - (b8 >> 3)) * 8 + (b8 & 7);
  const int rv0 = blockIdx.x * 256 + t;
  const bool writes_v = (int)blockIdx.x * 256 < n;
  if (bid >= ntiles && !writes_v) return;
  if (b8 >= 0 && bid < ntiles) {
    int I = (int)((sqrt(8.0 * bid + 1.0) - 1.0) * 0.5);
    while ((I + 1) * (I + 2) / 2 <= bid) ++I;
    while (I * (I + 1) / 2 > bid) --I;
    const int J = bid - I * (I + 1) / 2;
    const int r0 = TS * I, c0 = TS * J;
    const bool rok = r0 + lane < m;
    // wave-uniform column pointers with a per-lane row offset
    const int wu = __builtin_amdgcn_readfirstlane(wv);
    const double* base = A + (size_t)(o + r0) + (size_t)(o + c0 + wu) * ld;
    double x[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int c = c0 + wu + 4 * q;
      x[q] = (rok && c < m) ? base[(size_t)(4 * q) * ld + lane] : 0.0;
    }
    if (t < TS) {
      vr[t] = r0 + t < m ? a[o + r0 + t] : 0.0;
    } else if (t < 2 * TS) {
      vc[t - TS] = c0 + t - TS < m ? a[o + c0 + t - TS] : 0.0;
    }
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) s += x[q] * vc[wv + 4 * q];
    red[wv][lane] = s;
    if (I > J) {
      const double vl = vr[lane];
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q] *= vl;
      fold_halves<16, 32>(x, lane);
      const double z = fold_sum<2>(x[0]);
      const int c = c0 + wv + 4 * (lane >> 2);
      if ((lane & 3) == 0 && c < m) Ypart[(size_t)I * m + c] = z;
    }
    __syncthreads();
    if (wv == 0) {
      const double rowp = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
      if (r0 + lane < m) Ypart[(size_t)J * m + r0 + lane] = rowp;
      double pv = wave_sum(rowp * vr[lane]);
      if (lane == 0) pyv[bid] = (I > J ? 2.0 : 1.0) * pv;
    }
    if (!writes_v) return;
  }
  // the reflector: panel dots, v into the panel, d, e, tau, sc
  const double alpha = a[j + 1];
  const double av0 = (rv0 < n && rv0 > j + 1) ? a[rv0] : 0.0;
  const double ajj = (blockIdx.x == 0 && t == 0) ? a[j] : 0.0;
  const double a00 = (blockIdx.x == 0 && t == 0) ? A[(size_t)o + (size_t)o * ld] : 0.0;
  double xn2 = sum_partials(pnorm, npn, sh4);
  double beta = alpha, tv = 0.0, scale = 1.0;
  if (xn2 != 0.0) {
    beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
    tv = (beta - alpha) / beta;
    scale = 1.0 / (alpha - beta);
  }
  if (blockIdx.x == 0 && t == 0) {
    d[j] = ajj;
    e[j] = beta;
    tau[j] = tv;
    sc[0] = scale;
    sc[1] = a00;
  }
  for (int r = rv0; r < n; r += gridDim.x * 256) {
    double v = r <= j ? 0.0 : (r == j + 1 ? 1.0 : (r == rv0 ? av0 : a[r]) * scale);
    Vp[r + (size_t)i * ld] = v;
    V2[r + (size_t)i * ld] = v;
  }
  if ((int)blockIdx.x < i) {
    const int q = (int)blockIdx.x;
    const double* wq = Wp + (size_t)q * ld + o;
    const double* vq = Vp + (size_t)q * ld + o;
    const double* ac = a + o;
    double s0 = 0.0, s1 = 0.0, u0 = 0.0, u1 = 0.0;
    int l = t;
    // two rows per thread in flight
    for (; l + 256 < m; l += 2 * 256) {
      const double a0 = ac[l], a1 = ac[l + 256];
      const double w0 = wq[l], w1 = wq[l + 256];
      const double p0 = vq[l], p1 = vq[l + 256];
      const double v0 = l == 0 ? 1.0 : a0 * scale;
      const double v1 = a1 * scale;
      s0 += w0 * v0;
      u0 += w1 * v1;
      s1 += p0 * v0;
      u1 += p1 * v1;
    }
    for (; l < m; l += 256) {
      const double vv = l == 0 ? 1.0 : ac[l] * scale;
      s0 += wq[l] * vv;
      s1 += vq[l] * vv;
    }
    s0 = block_sum256(s0 + u0, sh4);
    s1 = block_sum256(s1 + u1, sh4);
    if (t == 0) {
      ab[q] = s0;
      ab[i + q] = s1;
    }
  }
}

// sum of p[b] over b = t (mod 256) for thread t, eight loads in flight
__device__ __forceinline__ double strided_partial(const double* __restrict__ p, int np, int t) {
  double q0 = 0.0, q1 = 0.0, q2 = 0.0, q3 = 0.0, q4 = 0.0, q5 = 0.0, q6 = 0.0, q7 = 0.0;
  int b = t;
  for (; b + 7 * 256 < np; b += 8 * 256) {
    q0 += p[b];
    q1 += p[b + 256];
    q2 += p[b + 512];
    q3 += p[b + 768];
    q4 += p[b + 1024];
    q5 += p[b + 1280];
    q6 += p[b + 1536];
    q7 += p[b + 1792];
  }
  for (; b < np; b += 256) q0 += p[b];
  return ((q0 + q1) + (q2 + q3)) + ((q4 + q5) + (q6 + q7));
}


constexpr int POST_ROWS = 16;   // rows per block of the post kernel

// Rows [r0, r0 + 16), r0 = 16 (b0 + blockIdx.x), b0 = (j + 1) / 16 (rows up
// to j are finished): w = tau (y - V a - W b) + alpha v, v -> A(:, j), the
// next panel column's update and its squared-tail partial sum. Thread
// (row rr = t % 16, part = t / 16) sums its share t = part (mod 16) of the
// symv row partials and q = part (mod 16) of the panel terms; the 16 parts
// meet in LDS once. The symv partials are of A22 a; with the reflector's
// scale s = sc[0] and beta = e[j], y(r) = s ((A22 a)(r) - beta A(r, j+1)),
// and v^T A22 v = s^2 (a^T A22 a - 2 beta (A22 a)(0) + beta^2 sc[1]),
// sc[1] = A(j+1, j+1). The scalars (v^T A22 v, a^T b, y(j+1), the panel
// dot at j+1) are formed the same way in every block, so all blocks agree
// bit for bit.
__global__ __launch_bounds__(256) void trd_post_kernel(
    double* __restrict__ A, int n, int j, int i, int nsym, const double* __restrict__ Vp,
    double* __restrict__ Wp, const double* __restrict__ Ypart, int T,
    const double* __restrict__ ab, const double* __restrict__ pyv,
    const double* __restrict__ tau, const double* __restrict__ e,
    const double* __restrict__ sc, int next, double* __restrict__ pnorm, int b0) {
  __shared__ double red[3][POST_ROWS][POST_ROWS + 1];
  __shared__ double scr[4][4];
  const size_t ld = (size_t)n;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int rr = t % POST_ROWS, part = t / POST_ROWS;
  const int r = (b0 + (int)blockIdx.x) * POST_ROWS + rr;
  const int jn = j + 1;
  const int m = n - j - 1;
  const bool live = r > j && r < n;   // rows of v, w and the update
  // symv row partials: y(r) = sum_t Ypart[t][r - jn]
  double yp = 0.0;
  if (live) {
    const double* yc = Ypart + (r - jn);
    double q0 = 0.0, q1 = 0.0, q2 = 0.0, q3 = 0.0;
    int tt = part;
    for (; tt + 3 * POST_ROWS < T; tt += 4 * POST_ROWS) {
      q0 += yc[(size_t)tt * m];
      q1 += yc[(size_t)(tt + POST_ROWS) * m];
      q2 += yc[(size_t)(tt + 2 * POST_ROWS) * m];
      q3 += yc[(size_t)(tt + 3 * POST_ROWS) * m];
    }
    for (; tt < T; tt += POST_ROWS) q0 += yc[(size_t)tt * m];
    yp = (q0 + q1) + (q2 + q3);
  }
  // panel terms over q < i: V(r,q) a_q + W(r,q) b_q and, for the next
  // column, V(r,q) W(jn,q) + W(r,q) V(jn,q)
  double sw = 0.0, sn = 0.0;
  if (live) {
    for (int q = part; q < i; q += POST_ROWS) {
      const double vq = Vp[r + (size_t)q * ld], wq = Wp[r + (size_t)q * ld];
      sw += vq * ab[q] + wq * ab[i + q];
      if (next) sn += vq * Wp[jn + (size_t)q * ld] + wq * Vp[jn + (size_t)q * ld];
    }
  }
  // block scalars: every thread a strided share of the v^T A22 v partials;
  // wave 1: y(jn); wave 2: a^T b; wave 3: the panel dot at row jn
  double pv = strided_partial(pyv, nsym, t);
  double s1 = 0.0;
  if (wv == 1) {
    for (int tt = lane; tt < T; tt += 64) s1 += Ypart[(size_t)tt * m];
  } else if (wv == 2) {
    if (lane < i) s1 = ab[lane] * ab[i + lane];
  } else if (wv == 3) {
    if (next && lane < i)
      s1 = Vp[jn + (size_t)lane * ld] * ab[lane] + Wp[jn + (size_t)lane * ld] * ab[i + lane];
  }
  // wave 0's operands of the final step, loaded before the barrier
  const double tj = tau[j], bj = e[j], sj = sc[0], a00 = sc[1];
  double vr0 = 0.0, ajn0 = 0.0;
  if (wv == 0 && lane < POST_ROWS && r < n) {
    vr0 = Vp[r + (size_t)i * ld];
    if (r >= jn) ajn0 = A[r + (size_t)jn * ld];
  }
  pv = wave_sum(pv);
  s1 = wave_sum(s1);
  red[0][part][rr] = yp;
  red[1][part][rr] = sw;
  red[2][part][rr] = sn;
  if (lane == 0) {
    scr[0][wv] = pv;
    scr[1][wv] = s1;
  }
  __syncthreads();
  if (wv != 0) return;
  const double ata = (scr[0][0] + scr[0][1]) + (scr[0][2] + scr[0][3]);
  const double y0a = scr[1][1], atb = scr[1][2], djn = scr[1][3];
  const double ytv = sj * sj * ((ata - 2.0 * bj * y0a) + bj * bj * a00);
  const double y0 = sj * (y0a - bj * a00);
  const double alpha = -0.5 * tj * tj * (ytv - 2.0 * atb);
  double s = 0.0;
  if (lane < POST_ROWS && r < n) {
    double ya = 0.0, swr = 0.0, snr = 0.0;
#pragma unroll
    for (int p = 0; p < POST_ROWS; ++p) {
      ya += red[0][p][lane];
      swr += red[1][p][lane];
      snr += red[2][p][lane];
    }
    const double yr = sj * (ya - bj * ajn0);
    const double vr = vr0;
    double wr = 0.0;
    if (r > j && tj != 0.0) wr = tj * (yr - swr) + alpha * vr;
    Wp[r + (size_t)i * ld] = wr;
    if (r > j) A[r + (size_t)j * ld] = vr;
    if (next && r >= jn) {
      // w(jn) for the panel column i (V(jn, i) = 1)
      const double wj1 = (tj != 0.0) ? tj * (y0 - djn) + alpha : 0.0;
      double acc = ajn0 - snr;
      acc -= vr * wj1 + wr;
      A[r + (size_t)jn * ld] = acc;
      if (r >= jn + 2) s = acc * acc;
    }
  }
  if (next) {
    s = wave_sum(s);
    if (lane == 0) pnorm[b0 + blockIdx.x] = s;
  }
}

// trailing blocks this small are reduced by one workgroup: 192 x 192 doubles
// are 144 of a thread's 256 registers; 256 rows would not fit
constexpr int TRD_TAIL = 192;

// The trailing block of m = n - p <= 32 RB rows and columns (every earlier
// update applied, its lower triangle current) reduced to tridiagonal form by
// one 512-thread workgroup, column by column (dsytd2): y = tau A22 v,
// w = y - tau/2 (y^T v) v, A22 -= v w^T + w v^T. d, e, tau and the
// reflectors (v(j+1) = 1 stored) go where the per-column kernels put them.
//
// Bound: the latency of a column's serial chain. The block stays in
// registers (both triangles): thread (i, c), i = lane % 32, c = 2 wave +
// lane / 32, holds rows i + 32 a, a < RB, of columns c + 16 b, b < 2 RB. The
// columns are taken 32 at a time (phase RA: rows and columns from 32 RA on
// are live), so that the code of a phase has no tests for finished blocks. A
// column lies in one half-wave, so its norm is a half-wave sum; A22 v is
// formed as column sums (the block is symmetric), a lane's partials first
// halved by one exchange between the half-wave's two rows of 16 lanes; only
// v, y and the partials of y^T v pass through LDS, two barriers per column.
// 192 columns take 0.34 ms, 1.8 us each (two launches a column before: 8.5;
// the LDS-resident tail of 128 rows, eight barriers a column: 5.7).
template <int RB>
struct TrdTail {
  static constexpr int CB = 2 * RB;
  double* A;
  double *d, *e, *tau;
  double *vs, *ys, *part, *scal;   // LDS: 2 x 32 RB, 2 x 32 RB, 2 x 8, 2
  int n, p, m, lane, wave, i, c;
  bool up;
  double x[RB][CB];

  template <int RA>
  __device__ __forceinline__ void phase() {
    constexpr int CA = 2 * RA, NC = CB - CA, NR = RB - RA;   // live blocks
    const int k1 = min(m - 1, 32 * RA + 32);
    for (int k = 32 * RA; k < k1; ++k) {
      const int buf = k & 1;
      double* v = vs + buf * 32 * RB;
      double* y = ys + buf * 32 * RB;
      if (c == (k & 15)) {
        // this half-wave holds column k: block CA or CA + 1
        const bool hi = (k & 16) != 0;
        double col[RB];
#pragma unroll
        for (int a = RA; a < RB; ++a) col[a] = hi ? x[a][CA + 1] : x[a][CA];
        double s = 0.0, al = 0.0;
#pragma unroll
        for (int a = RA; a < RB; ++a) {
          const int r = i + 32 * a;
          if (r > k + 1) s += col[a] * col[a];
          if (a == ((k + 1) >> 5)) al = col[a];
        }
        const double alpha = __shfl(al, (lane & 32) | ((k + 1) & 31), 64);
        const double xn2 = fold_sum<16>(s);
        double beta = alpha, tv = 0.0, scale = 1.0;
        if (xn2 != 0.0) {
          beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
          tv = (beta - alpha) / beta;
          scale = 1.0 / (alpha - beta);
        }
#pragma unroll
        for (int a = RA; a < RB; ++a) {
          const int r = i + 32 * a;
          const double vr = r <= k ? 0.0 : (r == k + 1 ? 1.0 : col[a] * scale);
          v[r] = vr;
          if (r > k && r < m) A[(size_t)(p + r) + (size_t)(p + k) * n] = vr;
        }
        if (i == 0) {
          e[p + k] = beta;
          tau[p + k] = tv;
          scal[buf] = tv;
        }
        if (i == (k & 31)) d[p + k] = col[RA];
      }
      __syncthreads();
      const double tv = scal[buf];
      double vr[NR], vc[NC];
#pragma unroll
      for (int a = 0; a < NR; ++a) vr[a] = v[i + 32 * (RA + a)];
#pragma unroll
      for (int b = 0; b < NC; ++b) vc[b] = v[c + 16 * (CA + b)];
      // y(q) = sum_r A(r, q) v(r); rows up to k have v = 0
      double s[NC];
#pragma unroll
      for (int b = 0; b < NC; ++b) {
        s[b] = 0.0;
#pragma unroll
        for (int a = 0; a < NR; ++a) s[b] += x[RA + a][CA + b] * vr[a];
      }
      // lanes with bit 4 clear end up with the first half of the columns
      double pv = 0.0;
#pragma unroll
      for (int b = 0; b < NR; ++b) {
        const double z = row16_sum(swap_add<16>(s[b], s[b + NR]));
        if ((i & 15) == b) y[c + 16 * (CA + b + (up ? NR : 0))] = z;
        pv += z * (up ? vc[b + NR] : vc[b]);
      }
      pv = swap_add<16>(pv, pv);
      pv = swap_add<32>(pv, pv);
      if (lane == 0) part[buf * 8 + wave] = pv;
      __syncthreads();
      double ytv = 0.0;
#pragma unroll
      for (int q = 0; q < 8; ++q) ytv += part[buf * 8 + q];
      const double f = -0.5 * tv * tv * ytv;
      double wr[NR], wc[NC];
#pragma unroll
      for (int a = 0; a < NR; ++a) wr[a] = tv * y[i + 32 * (RA + a)] + f * vr[a];
#pragma unroll
      for (int b = 0; b < NC; ++b) wc[b] = tv * y[c + 16 * (CA + b)] + f * vc[b];
      // finished rows and columns (up to k) have v = 0 but not w; nothing
      // reads them again
#pragma unroll
      for (int b = 0; b < NC; ++b)
#pragma unroll
        for (int a = 0; a < NR; ++a)
          x[RA + a][CA + b] -= vr[a] * wc[b] + wr[a] * vc[b];
    }
    if constexpr (RA + 1 < RB)
      if (k1 < m - 1) phase<RA + 1>();
  }
};

template <int RB>
__global__ __launch_bounds__(512) void trd_tail_kernel(double* __restrict__ A, int n, int p,
                                                       double* __restrict__ d,
                                                       double* __restrict__ e,
                                                       double* __restrict__ tau) {
  __shared__ double sh[2 * 32 * RB + 2 * 32 * RB + 2 * 8 + 2];
  TrdTail<RB> q;
  q.A = A;
  q.d = d;
  q.e = e;
  q.tau = tau;
  q.vs = sh;
  q.ys = sh + 64 * RB;
  q.part = sh + 128 * RB;
  q.scal = sh + 128 * RB + 16;
  q.n = n;
  q.p = p;
  q.m = n - p;
  q.lane = threadIdx.x & 63;
  q.wave = threadIdx.x >> 6;
  q.i = q.lane & 31;
  q.c = 2 * q.wave + (q.lane >> 5);
  q.up = (q.lane & 16) != 0;
#pragma unroll
  for (int b = 0; b < 2 * RB; ++b)
#pragma unroll
    for (int a = 0; a < RB; ++a) {
      const int r = q.i + 32 * a, c = q.c + 16 * b;
      const int hi = r > c ? r : c, lo = r > c ? c : r;
      q.x[a][b] = hi < q.m ? A[(size_t)(p + hi) + (size_t)(p + lo) * n] : 0.0;
    }
  q.template phase<0>();
  const int l = q.m - 1;
  if (q.c == (l & 15) && q.i == (l & 31)) {
    double dl = 0.0;
#pragma unroll
    for (int b = 0; b < 2 * RB; ++b)
      if (b == (l >> 4)) dl = q.x[b / 2][b];
    d[n - 1] = dl;
    tau[n - 1] = 0.0;
  }
}

// -------------------------------------------- resident reduction (m <= 3584)
// The trailing block of m = n - p <= 512 K rows and columns (every earlier
// update applied, its lower triangle current) reduced by `cols` columns by
// workgroups that keep it in registers: workgroup g owns rows R g .. R g + R - 1
// (whole rows, both triangles; R = 16; K = 6 has 12, which the registers still
// hold, K = 7 has 14, RL = 4 of them in LDS), thread t of 512 columns t + 512 k,
// k < K.
//
// Bound: the latency of one exchange per column between the workgroups (write
// to memory, poll, read); the rest is the chain of
// three barriers and two sums over the block. The chip-wide kernels pay two
// launches and three dependent passes over memory per column instead. A column
// takes 2.8, 3.4, 4.2, 4.9 us for K = 1, 2, 3, 4 (8.2 to 13 before; 0.3 more
// where the slot is emptied before the column and not while its exchange is
// under way); whole eigendecompositions: n = 512 3.7 -> 1.9 ms, 1000 8.3 -> 4.1,
// 2048 20.4 -> 10.1, 3000 23.5 -> 18.4 by K = 6, 4096 40.0 -> 36.2 by K = 7. A
// workgroup's values go out as one store: one by one, by the lane that holds
// them, took 15% longer.
//
// Column j, every workgroup alike: from a = A(:, j) (known to all) the norm,
// the reflector v and tau; one pass over the workgroup's rows applies the
// previous column's A -= v w^T + w v^T and forms y = A v; the workgroup
// publishes y(r) and A(r, j + 1) for its rows, and reads both for all rows.
// Then w = tau y - tau^2/2 (y^T v) v, and the next column is A(:, j + 1) -
// v w(j+1) - w v(j+1): one exchange gives all that the next column needs, and
// every workgroup computes the same bits from it.
//
// The exchange is data that validates itself: a slot holds MID_EMPTY until its
// value is there (a result with these very bits is published with the last bit
// flipped; both are NaNs). Four slots take turns: at column j a workgroup
// empties its part of slot (j + 2) mod 4, last used at column j - 2; all that
// read that have published column j - 1 since, which was gathered before.
// Values go through agent-scope atomics (past the L2 of the XCD); the emptying
// stores are waited for before the barrier that comes before the next column
// is published, so whoever has seen that one sees them. A workgroup whose rows
// are done leaves before it would gather (nothing waits for it any more).
//
// All workgroups have to be resident at once: at most 256, one per CU. The
// host lets one such reduction run at a time on a device. Against other
// processes on it every wait is bounded by `limit` ticks (100 MHz): then
// *stop is set, every workgroup leaves, and the host starts over without this
// kernel.
constexpr int MID_MAX = 3584;
constexpr size_t MID_LDS = 4 * 3584 * sizeof(double);
constexpr unsigned long long MID_EMPTY = 0x7FF8A5A5C3C35A5AULL;
typedef unsigned long long mid_t;

__device__ __forceinline__ mid_t mid_get(const mid_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void mid_put(mid_t* p, mid_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void trd_mid_clear_kernel(mid_t* ring, int count, int* stop, bool first) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e < count) ring[e] = MID_EMPTY;
  if (e == 0 && first) *stop = 0;
}

template <int K, int RV, int RL>
__global__ __launch_bounds__(512) void trd_mid_kernel(double* __restrict__ A, int n, int p, int cols,
                                                      double* __restrict__ d,
                                                      double* __restrict__ e,
                                                      double* __restrict__ tau, mid_t* ring,
                                                      int* stop, long long limit) {
  constexpr int MP = 512 * K, R = RV + RL;
  extern __shared__ double trd_mid_lds[];   // rows RV .. R - 1, MP each
  __shared__ double red1[8], red2[8], part[8][16], ncol[R], rv[R], rw[R], sc[2];
  __shared__ int bad;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int m = n - p, row0 = (int)blockIdx.x * R;
  const bool writer = blockIdx.x + 1 == gridDim.x;   // its rows are the last ones done
  double* Ap = A + (size_t)p * n + p;
  double x[K][RV];
  double* xl = trd_mid_lds + t;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = t + 512 * k;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = row0 + i, hi = r > c ? r : c, lo = r > c ? c : r;
      const double q = hi < m ? Ap[(size_t)lo * n + hi] : 0.0;
      if (i < RV) x[k][i < RV ? i : 0] = q;
      else xl[(i - RV) * MP + 512 * k] = q;
    }
  }
  // a: column j; v, w: column j - 1's until the pass, then j's
  double a[K], v[K], w[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = t + 512 * k;
    a[k] = c < m ? Ap[c] : 0.0;
    v[k] = w[k] = 0.0;
  }
  if (t < R) rv[t] = rw[t] = 0.0;
  if (t == 0) bad = 0;
  for (int j = 0; j < cols; ++j) {
    mid_t* slot = ring + (j & 3) * 2 * MP;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = t + 512 * k;
      if (c >= j + 2) s += a[k] * a[k];   // a is 0 from m on
      if (c == j + 1) sc[0] = a[k];
    }
    s = wave_sum(s);
    if (lane == 0) red1[wv] = s;
    __syncthreads();
    const double alpha = sc[0];
    const double xn2 = ((red1[0] + red1[1]) + (red1[2] + red1[3])) +
                       ((red1[4] + red1[5]) + (red1[6] + red1[7]));
    double beta = alpha, tv = 0.0, scale = 1.0;
    if (xn2 != 0.0) {
      beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
      tv = (beta - alpha) / beta;
      scale = 1.0 / (alpha - beta);
    }
    double vn[K], y[16];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = t + 512 * k;
      vn[k] = c <= j ? 0.0 : c == j + 1 ? 1.0 : a[k] * scale;
      if (writer && c == j) d[p + j] = a[k];
    }
    if (writer && t == 0) {
      e[p + j] = beta;
      tau[p + j] = tv;
    }
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const double pr = rv[i], qr = rw[i];
      y[i] = 0.0;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        x[k][i] -= pr * w[k] + qr * v[k];
        y[i] += x[k][i] * vn[k];
      }
    }
#pragma unroll
    for (int i = RV; i < R; ++i) {
      const double pr = rv[i], qr = rw[i];
      y[i] = 0.0;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        double q = xl[(i - RV) * MP + 512 * k];
        q -= pr * w[k] + qr * v[k];
        xl[(i - RV) * MP + 512 * k] = q;
        y[i] += q * vn[k];
      }
    }
    if (t == ((j + 1) & 511)) {
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (k == (j + 1) / 512) {
#pragma unroll
          for (int i = 0; i < RV; ++i) ncol[i] = x[k][i];
#pragma unroll
          for (int i = RV; i < R; ++i) ncol[i] = xl[(i - RV) * MP + 512 * k];
        }
    }
#pragma unroll
    for (int i = R; i < 16; ++i) y[i] = 0.0;
    fold_halves<16, 32>(y, lane);
    const double z = fold_sum<2>(y[0]);
    if ((lane & 3) == 0) part[wv][lane >> 2] = z;
    __syncthreads();
    if (t < 2 * R) {
      const int i = t % R, r = row0 + i;
      double q = ncol[i];
      if (t < R)
        q = ((part[0][i] + part[1][i]) + (part[2][i] + part[3][i])) +
            ((part[4][i] + part[5][i]) + (part[6][i] + part[7][i]));
      if (r > j && r < m) {
        mid_t b = (mid_t)__double_as_longlong(q);
        if (b == MID_EMPTY) b ^= 1;
        mid_put(slot + (t / R) * MP + r, b);
      }
    }
    // two columns ahead: done, and past a barrier, before the next column is
    // published
    if (wv == 7 && lane < 2 * R && row0 + lane % R > j && row0 + lane % R < m)
      mid_put(ring + ((j + 2) & 3) * 2 * MP + (lane / R) * MP + row0 + lane % R, MID_EMPTY);
    // whole workgroup: no row after j + 1 and none to hand back
    if (row0 + R - 1 <= j + 1 && row0 + R - 1 < cols) return;
    mid_t yb[K], ab[K];
    {
      long long t0 = 0;
      for (int spins = 0;; ++spins) {
        bool all = true;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int c = t + 512 * k;
          yb[k] = ab[k] = 0;
          if (c > j && c < m) {
            yb[k] = mid_get(slot + c);
            ab[k] = mid_get(slot + MP + c);
            all = all && yb[k] != MID_EMPTY && ab[k] != MID_EMPTY;
          }
        }
        if (all) break;
        if (spins == 0) t0 = wall_clock64();
        if ((spins & 63) == 63 || limit == 0) {
          if (__hip_atomic_load(stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
              wall_clock64() - t0 >= limit) {
            __hip_atomic_store(stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bad = 1;
            break;
          }
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the emptying stores
    double g = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = t + 512 * k;
      v[k] = vn[k];
      w[k] = __longlong_as_double((long long)yb[k]);
      a[k] = __longlong_as_double((long long)ab[k]);
      g += c > j ? w[k] * v[k] : 0.0;
      if (c == j + 1) sc[1] = w[k];
    }
    g = wave_sum(g);
    if (lane == 0) red2[wv] = g;
    __syncthreads();
    if (bad) return;   // whole workgroup
    if (writer) {
      // only now, past the barrier: every workgroup has published, so has
      // read the column that is overwritten
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int c = t + 512 * k;
        if (c > j && c < m) Ap[(size_t)j * n + c] = v[k];
      }
    }
    const double ytv = ((red2[0] + red2[1]) + (red2[2] + red2[3])) +
                       ((red2[4] + red2[5]) + (red2[6] + red2[7]));
    const double f = -0.5 * tv * tv * ytv, w1 = tv * sc[1] + f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = t + 512 * k;
      w[k] = c > j ? tv * w[k] + f * v[k] : 0.0;
      a[k] = c > j ? a[k] - (v[k] * w1 + w[k]) : 0.0;
      if (c >= row0 && c < row0 + R) {
        rv[c - row0] = v[k];
        rw[c - row0] = w[k];
      }
    }
  }
  __syncthreads();
  // the last update, and the rest back: row r's part right of the diagonal
  // into column r
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = row0 + i;
    const double pr = rv[i], qr = rw[i];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = t + 512 * k;
      if (r >= cols && c >= r && c < m)
        Ap[(size_t)r * n + c] = (i < RV ? x[k][i < RV ? i : 0] : xl[(i - RV) * MP + 512 * k]) -
                                (pr * w[k] + qr * v[k]);
    }
  }
}

// A's rows and columns from p on, to or from a copy
__global__ void trd_copy_kernel(double* __restrict__ A, int n, int p, double* __restrict__ B,
                                bool back) {
  const int m = n - p;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < (int64_t)m * m;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(q % m), c = (int)(q / m);
    double* x = A + (size_t)(p + c) * n + p + r;
    if (back) *x = B[q];
    else B[q] = *x;
  }
}

__global__ void trd_last_kernel(const double* __restrict__ A, int n, double* d, double* tau) {
  d[n - 1] = A[(size_t)(n - 1) * n + (n - 1)];
  tau[n - 1] = 0.0;
}

// --------------------------------------------------------- back-transform
// reflector j has v(j+off) = 1 and v(r) = A[r, j] below it (off = 1 for the
// tridiagonal reduction, 0 for QR)
__global__ void bt_build_v_kernel(const double* __restrict__ A, int n, int p, int nbp, int off,
                                  double* __restrict__ Vb) {
  int64_t tot = (int64_t)n * nbp;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int r = (int)(e % n), i = (int)(e / n);
    int j = p + i;
    double v = 0.0;
    if (r == j + off) v = 1.0;
    else if (r > j + off) v = A[r + (size_t)j * n];
    Vb[e] = v;
  }
}

// compact-WY triangular factor, forward columnwise (dlarft 'F','C'); G and
// tau are staged in LDS first so the column recurrence touches no HBM
__global__ void bt_larft_kernel(int nbp, const double* __restrict__ G, const double* __restrict__ tau,
                                double* __restrict__ T) {
  __shared__ double Ts[NB][NB + 1];
  __shared__ double Gs[NB][NB + 1];
  __shared__ double ts[NB];
  __shared__ double tmp[NB];
  int l = threadIdx.x;
  for (int e = l; e < NB * NB; e += blockDim.x) {
    int r = e % NB, c = e / NB;
    Ts[r][c] = 0.0;
    Gs[r][c] = (r < nbp && c < nbp) ? G[r + c * nbp] : 0.0;
  }
  if (l < nbp) ts[l] = tau[l];
  __syncthreads();
  for (int i = 0; i < nbp; ++i) {
    if (l < i) tmp[l] = -ts[i] * Gs[l][i];
    __syncthreads();
    if (l < i) {
      double s = 0.0;
      for (int m = l; m < i; ++m) s += Ts[l][m] * tmp[m];
      Ts[l][i] = s;
    }
    if (l == i) Ts[i][i] = ts[i];
    __syncthreads();
  }
  for (int e = l; e < nbp * nbp; e += blockDim.x) T[e] = Ts[e % nbp][e / nbp];
}

// After the tridiagonalisation column j of A holds v_j below the diagonal
// (v_j(j+1) = 1 stored); clearing rows 0..j makes A[:, p..p+NB) the panel's
// reflector block V with no copy.
__global__ void bt_clear_upper_kernel(double* __restrict__ A, int n) {
  int64_t tot = (int64_t)n * n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int r = (int)(e % n), j = (int)(e / n);
    if (r <= j) A[e] = 0.0;
  }
}

// Back-transform of a group of up to BT_GROUP consecutive reflectors at once:
// with Y = V^T U (the group's rows of U) and G = V^T V, U <- H_0 .. H_{b-1} U =
// U - V X, X = T Y, where T is never formed: T^-1 = diag(1 / tau) + the strict
// upper triangle of G (forward columnwise compact WY, any tau), so that
// X_i = tau_i (Y_i - sum_{q>i} G(i, q) X_q).
//
// One workgroup per 16 columns of U, 16 rows of X a step, last to first: the
// later rows' terms on MFMA, their k split over the four waves, then the
// 16 x 16 triangle by its inverse (T of the 16 reflectors), formed beforehand
// for all steps at once. Bound by latency: everything is loaded up front (the
// fragments of G in registers) and a step is three barriers. 128 reflectors:
// 14 us for 100 columns, 15 for 1000; with 32-row steps of dot products in LDS
// and T formed by a kernel of its own 17 and 23, and for that kernel 46 (n =
// 200) to 216 (n = 2048).
constexpr int BT_GROUP = 128;
typedef double btv_t __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void bt_group_solve_kernel(int nbg, int k,
                                                             const double* __restrict__ Y,
                                                             const double* __restrict__ Gg,
                                                             const double* __restrict__ tau,
                                                             double* __restrict__ X2) {
  constexpr int S = BT_GROUP / 16;
  __shared__ double gs[S][257], Ts[S][16][17], xs[BT_GROUP][16], part[4][256], xt[256];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int lr = lane & 15, lg = lane >> 4, ti = t & 15, tc = t >> 4;
  const int c = (int)blockIdx.x * 16 + tc;
  btv_t f[S - 1][2];   // wave wv's fragments of G, S - 1 - b of step b used
  double y[S];
#pragma unroll
  for (int b = 0; b < S; ++b) {
    const int r = 16 * b + ti, q = 16 * b + tc;
    y[b] = (c < k && r < nbg) ? Y[(size_t)c * nbg + r] : 0.0;
    double g = 0.0;
    if (ti < tc && q < nbg) g = Gg[r + (size_t)q * nbg];
    if (ti == tc && q < nbg) g = tau[q];
    gs[b][ti + 16 * tc] = g;
  }
#pragma unroll
  for (int b = 0; b < S - 1; ++b)
#pragma unroll
    for (int u = 0; u < S - 1 - b; ++u) {
      const int r = 16 * b + lr, q = 16 * (b + 1) + 4 * (wv + 4 * u) + lg;
      f[b][u / 4][u % 4] = (r < nbg && q < nbg) ? Gg[r + (size_t)q * nbg] : 0.0;
    }
  __syncthreads();
  if (t < 16 * S) {
    // column ti of step tc's T
    const double* g = gs[tc];
    double x[16];
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      const double ta = g[i + 16 * i];
      double s = 0.0;
#pragma unroll
      for (int q = i + 1; q < 16; ++q) s += g[i + 16 * q] * x[q];
      x[i] = i == ti ? ta : -ta * s;
      if (i > ti) x[i] = 0.0;
      Ts[tc][i][ti] = x[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = S - 1; b >= 0; --b) {
    double x = y[b];
    if (b < S - 1) {
      btv_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < S - 1 - b; ++u)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(
            f[b][u / 4][u % 4], xs[16 * (b + 1) + 4 * (wv + 4 * u) + lg][lr], acc, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wv][4 * r + lg + 16 * lr] = acc[r];
      __syncthreads();
      x -= (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    }
    xt[t] = x;
    __syncthreads();
    if (wv == 0) {
      btv_t d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(Ts[b][lr][4 * q + lg], xt[4 * q + lg + 16 * lr], d,
                                                 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) xs[16 * b + 4 * r + lg][lr] = d[r];
    }
    __syncthreads();
  }
  if (c >= k) return;
#pragma unroll
  for (int b = 0; b < S; ++b)
    if (16 * b + ti < nbg) X2[(size_t)c * nbg + 16 * b + ti] = xs[16 * b + ti][tc];
}

// tau of every reflector from the panels' compact-WY factors (their diagonals)
__global__ void bt_tau_kernel(const double* __restrict__ Tall, int nrefl, double* __restrict__ tau) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nrefl) return;
  const int p = i / NB, nb = min(NB, nrefl - p * NB);
  tau[i] = Tall[(size_t)p * NB * NB + (size_t)(i % NB) * (nb + 1)];
}

// --------------------------------------------------------- divide & conquer
// Q = Qn = 0: the leaves and every merge write whole block squares, and entries
// outside the current squares of both ping-pong buffers must stay zero
__global__ void dc_init_kernel(int n, double* Q, double* Qn) {
  int64_t tot = (int64_t)n * n;
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < tot;
       x += (int64_t)gridDim.x * blockDim.x) {
    Q[x] = 0.0;
    Qn[x] = 0.0;
  }
}

__device__ void bitonic_sort(double* key, int* val, int np2) {
  for (int k = 2; k <= np2; k <<= 1) {
    for (int jj = k >> 1; jj > 0; jj >>= 1) {
      for (int i = threadIdx.x; i < np2; i += blockDim.x) {
        int ixj = i ^ jj;
        if (ixj > i) {
          bool up = ((i & k) == 0);
          double a = key[i], b = key[ixj];
          if ((a > b) == up) {
            key[i] = b;
            key[ixj] = a;
            int tv = val[i];
            val[i] = val[ixj];
            val[ixj] = tv;
          }
        }
      }
      __syncthreads();
    }
  }
}

struct DcBufs {
  double *zs, *dl, *wv, *dval, *rcs, *tau, *zh, *mrho;
  int *gcol, *dcol, *rcol, *org, *meta;
};

constexpr int DC_ZLDS = 4096;   // largest merge whose z is staged in LDS

__global__ __launch_bounds__(1024) void dc_prepare_kernel(int n, int s_lvl, int half,
                                                          const double* __restrict__ D,
                                                          const double* __restrict__ Q,
                                                          const double* __restrict__ e, DcBufs b) {
  extern __shared__ double lds_d[];
  int m = blockIdx.x;
  int r0 = m * s_lvl;
  int s = min(s_lvl, n - r0);
  if (s <= half) return;
  int s1 = half;
  int np2 = 1;
  while (np2 < s) np2 <<= 1;
  double* key = lds_d;
  int* val = (int*)(key + np2);
  for (int i = threadIdx.x; i < np2; i += blockDim.x) {
    key[i] = i < s ? D[r0 + i] : INFINITY;
    val[i] = r0 + (i < s ? i : 0);
  }
  __syncthreads();
  bitonic_sort(key, val, np2);
  double beta = e[r0 + s1 - 1];
  double sg = beta >= 0.0 ? 1.0 : -1.0;
  // z is in LDS when it fits beside d and the columns (s_lvl <= DC_ZLDS)
  double* z = s_lvl <= DC_ZLDS ? (double*)(val + np2) : b.zs + r0;
  for (int i = threadIdx.x; i < s; i += blockDim.x) {
    int c = val[i];
    double zi = (c < r0 + s1) ? Q[(size_t)c * n + (r0 + s1 - 1)] : sg * Q[(size_t)c * n + (r0 + s1)];
    z[i] = zi * 0.7071067811865476;
  }
  __syncthreads();
  __shared__ int ksh, serial, isum[16];
  __shared__ double wsum[16], amax[2][16];
  const double rho = 2.0 * fabs(beta);
  if (s_lvl <= DC_ZLDS) {
    // Entries with rho |z| <= tol are dropped, the others kept, both in sorted
    // order (a compaction). Consecutive kept entries that nearly coincide are
    // rotated into one, which carries N = sum d z^2 and Z2 = sum z^2 of its
    // run: whether an entry joins the run before it is a chain, but only that.
    // If some pair of neighbours calls for it by its own values, one thread
    // walks the kept entries for these decisions (a few multiply-adds each);
    // lists, rotations, square roots and divisions are formed by all threads
    // from the sums it leaves, with the ranks from prefix sums. The rules are
    // dc_deflate's. With that pass in one thread altogether 128 to 200 rows took
    // 39 us, the merges of a 4096-row density matrix 240 on average; now 20 and
    // 117 (most of it the sort and the walk).
    constexpr int ROT = 1 << 30;        // flag on kidx: joins the run before it
    int* kidx = (int*)(z + np2);
    int* rpre = kidx + np2;             // rotated entries before kept entry p
    double* runN = b.tau + r0;          // by kept entry; free until the roots
    double* runZ = b.zh + r0;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    double dm = 0.0, zm = 0.0;
    for (int i = t; i < s; i += blockDim.x) {
      dm = fmax(dm, fabs(key[i]));
      zm = fmax(zm, fabs(z[i]));
    }
    for (int o = 32; o > 0; o >>= 1) {
      dm = fmax(dm, __shfl_xor(dm, o, 64));
      zm = fmax(zm, __shfl_xor(zm, o, 64));
    }
    if (lane == 0) {
      amax[0][wv] = dm;
      amax[1][wv] = zm;
    }
    if (t == 0) serial = 0;
    __syncthreads();
    dm = 0.0;
    zm = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) {
      dm = fmax(dm, amax[0][q]);
      zm = fmax(zm, amax[1][q]);
    }
    const double tol = 8.0 * ITG_DC_EPS * fmax(dm, zm);
    // one test for the counts and the lists (NaN is kept): a list shorter
    // than its count would leave indices unset
    auto drops = [&](int i) { return rho * fabs(z[i]) <= tol; };
    // thread t owns the contiguous entries [t cs, t cs + cs)
    const int cs = (s + (int)blockDim.x - 1) / (int)blockDim.x;
    const int i0 = min(s, t * cs), i1 = min(s, i0 + cs);
    int cnt = 0;
    for (int i = i0; i < i1; ++i) cnt += drops(i) ? 0 : 1;
    // exclusive scan of the kept counts over the block
    int inc = cnt;
    for (int o = 1; o < 64; o <<= 1) {
      int u = __shfl_up(inc, o, 64);
      if (lane >= o) inc += u;
    }
    if (lane == 63) isum[wv] = inc;
    __syncthreads();
    int base = 0, total = 0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) {
      if (q < wv) base += isum[q];
      total += isum[q];
    }
    const int pos0 = base + inc - cnt;
    for (int i = i0, pos = pos0; i < i1; ++i)
      if (!drops(i)) kidx[pos++] = i;
    __syncthreads();
    for (int p = t + 1; p < total; p += blockDim.x) {
      const int pj = kidx[p - 1], j = kidx[p];
      double S = z[pj], Cc = z[j];
      double tau = sqrt(Cc * Cc + S * S);
      double tt = key[j] - key[pj];
      double it = 1.0 / tau;
      double c = Cc * it, sn = -S * it;
      if (fabs(tt * c * sn) <= tol) serial = 1;
    }
    __syncthreads();
    int nrot = 0;
    if (serial) {
      if (t == 0) {
        const double tol2 = tol * tol;
        int j = kidx[0];
        double dj = key[j], zj = z[j], N = dj * zj * zj, Z2 = zj * zj;
        runN[0] = N;
        runZ[0] = Z2;
        double dn = 0.0, zn = 0.0;
        int jn = 0;
        if (total > 1) {
          jn = kidx[1];
          dn = key[jn];
          zn = z[jn];
        }
        for (int p = 1; p < total; ++p) {
          j = jn;
          dj = dn;
          zj = zn;
          if (p + 1 < total) {   // the next entry's loads go out before this one's work
            jn = kidx[p + 1];
            dn = key[jn];
            zn = z[jn];
          }
          const double zj2 = zj * zj, T2 = Z2 + zj2, x = dj * Z2 - N;
          const bool rot = x * x * zj2 <= tol2 * Z2 * T2 * T2;
          N = rot ? N + dj * zj2 : dj * zj2;
          Z2 = rot ? T2 : zj2;
          if (rot) kidx[p] = j | ROT;
          runN[p] = N;
          runZ[p] = Z2;
        }
      }
      __syncthreads();
      const int cp = (total + (int)blockDim.x - 1) / (int)blockDim.x;
      const int p0 = min(total, t * cp), p1 = min(total, p0 + cp);
      int rc = 0;
      for (int p = p0; p < p1; ++p) rc += (kidx[p] & ROT) ? 1 : 0;
      int ri = rc;
      for (int o = 1; o < 64; o <<= 1) {
        int u = __shfl_up(ri, o, 64);
        if (lane >= o) ri += u;
      }
      if (lane == 63) isum[wv] = ri;
      __syncthreads();
      int rb = 0;
      for (int q = 0; q < (int)(blockDim.x >> 6); ++q) {
        if (q < wv) rb += isum[q];
        nrot += isum[q];
      }
      rb += ri - rc;
      for (int p = p0; p < p1; ++p) {
        rpre[p] = rb;
        rb += (kidx[p] & ROT) ? 1 : 0;
      }
      __syncthreads();
    }
    // dropped entries, among them in order the entries rotated away
    for (int i = i0, pos = pos0; i < i1; ++i) {
      if (!drops(i)) {
        ++pos;
        continue;
      }
      const int q = r0 + i - pos + (!serial ? 0 : pos < total ? rpre[pos] : nrot);
      b.dval[q] = key[i];
      b.dcol[q] = val[i];
    }
    for (int p = t; p < total; p += blockDim.x) {
      const bool rot = serial && (kidx[p] & ROT);
      const int j = kidx[p] & ~ROT, rp = serial ? rpre[p] : 0;
      if (rot) {
        const int pj = kidx[p - 1] & ~ROT;
        const bool single = !(kidx[p - 1] & ROT);
        const double it = 1.0 / sqrt(runZ[p]), c = z[j] * it;
        const double sn = -(single ? z[pj] : sqrt(runZ[p - 1])) * it;
        const double dp = single ? key[pj] : runN[p - 1] / runZ[p - 1];
        b.rcol[2 * r0 + 2 * rp] = val[pj];
        b.rcol[2 * r0 + 2 * rp + 1] = val[j];
        b.rcs[2 * r0 + 2 * rp] = c;
        b.rcs[2 * r0 + 2 * rp + 1] = sn;
        b.dval[r0 + j - p + rp] = dp * c * c + key[j] * sn * sn;
        b.dcol[r0 + j - p + rp] = val[pj];
      }
      if (p + 1 == total || !(serial && (kidx[p + 1] & ROT))) {
        const int q = r0 + p - rp - (rot ? 1 : 0);
        b.dl[q] = rot ? runN[p] / runZ[p] : key[j];
        b.wv[q] = rot ? sqrt(runZ[p]) : z[j];
        b.gcol[q] = val[j];
      }
    }
    if (t == 0) {
      ksh = total - nrot;
      b.meta[3 * m] = total - nrot;
      b.meta[3 * m + 1] = s - total + nrot;
      b.meta[3 * m + 2] = nrot;
      b.mrho[2 * m] = rho;
    }
  } else if (threadIdx.x == 0) {
    // z does not fit in LDS beside d: the whole pass in one thread
    int nd = 0, nrot = 0;
    int k = dc_deflate(s, key, z, val, rho, b.dl + r0, b.wv + r0, b.gcol + r0, b.dval + r0,
                       b.dcol + r0, &nd, b.rcol + 2 * r0, b.rcs + 2 * r0, &nrot);
    ksh = k;
    b.meta[3 * m] = k;
    b.meta[3 * m + 1] = nd;
    b.meta[3 * m + 2] = nrot;
    b.mrho[2 * m] = rho;
  }
  __syncthreads();
  // sum of w^2 over the k kept entries: strided per thread, per wave, then
  // the 16 wave sums in order
  const int k = ksh;
  double w2 = 0.0;
  for (int j = threadIdx.x; j < k; j += blockDim.x) w2 += b.wv[r0 + j] * b.wv[r0 + j];
  for (int o = 32; o > 0; o >>= 1) w2 += __shfl_xor(w2, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = w2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += wsum[q];
    b.mrho[2 * m + 1] = t;
  }
}

__device__ __forceinline__ bool merge_range(int n, int s_lvl, int half, int m, int& r0, int& s) {
  r0 = m * s_lvl;
  s = min(s_lvl, n - r0);
  return s > half;
}

__global__ void dc_rotate_kernel(int n, int s_lvl, int half, double* __restrict__ Q, DcBufs b) {
  int m = blockIdx.x, r0, s;
  if (!merge_range(n, s_lvl, half, m, r0, s)) return;
  int nrot = b.meta[3 * m + 2];
  int r = r0 + blockIdx.y * blockDim.x + threadIdx.x;
  if (r >= r0 + s) return;
  for (int t = 0; t < nrot; ++t) {
    int pc = b.rcol[2 * r0 + 2 * t], qc = b.rcol[2 * r0 + 2 * t + 1];
    double c = b.rcs[2 * r0 + 2 * t], sn = b.rcs[2 * r0 + 2 * t + 1];
    double x = Q[(size_t)pc * n + r], yv = Q[(size_t)qc * n + r];
    Q[(size_t)pc * n + r] = c * x + sn * yv;
    Q[(size_t)qc * n + r] = c * yv - sn * x;
  }
}

// One wave per root: lanes split the sums over the k poles (the xor-butterfly
// sums leave every lane the same bits, so the iteration stays wave-uniform).
__global__ __launch_bounds__(256) void dc_secular_kernel(int n, int s_lvl, int half, DcBufs b) {
  int m = blockIdx.x, r0, s;
  if (!merge_range(n, s_lvl, half, m, r0, s)) return;
  int k = b.meta[3 * m];
  int lane = threadIdx.x & 63;
  int i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= k) return;
  const double* dl = b.dl + r0;
  const double* w = b.wv + r0;
  const double rho = b.mrho[2 * m];
  auto ev = [&](int o, double tau, int side, double* dpo, double* dpf, double* absum) {
    double f = 0.0, po = 0.0, pf = 0.0, ab = 0.0;
    const double dlo = dl[o];
    for (int j = lane; j < k; j += 64) {
      double del = (dl[j] - dlo) - tau;
      double t = w[j] / del;
      double term = rho * w[j] * t;
      f += term;
      ab += fabs(term);
      double dt = rho * t * t;
      bool origin_side = side > 0 ? (j <= o) : (j >= o);
      if (origin_side) po += dt; else pf += dt;
    }
    *dpo = wave_sum(po);
    *dpf = wave_sum(pf);
    *absum = 1.0 + wave_sum(ab);
    return 1.0 + wave_sum(f);
  };
  int o;
  double tv;
  dc_secular_root_with(i, k, dl, rho, b.mrho[2 * m + 1], ev, &o, &tv);
  if (lane == 0) {
    b.org[r0 + i] = o;
    b.tau[r0 + i] = tv;
  }
}

__device__ __forceinline__ double wave_prod(double v) {
  for (int o = 32; o > 0; o >>= 1) v *= __shfl_xor(v, o, 64);
  return v;
}

// zhat_i (Gu-Eisenstat, as dc_zhat) with one wave per i
__global__ __launch_bounds__(256) void dc_zhat_kernel(int n, int s_lvl, int half, DcBufs b) {
  int m = blockIdx.x, r0, s;
  if (!merge_range(n, s_lvl, half, m, r0, s)) return;
  int k = b.meta[3 * m];
  int lane = threadIdx.x & 63;
  int i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= k) return;
  const double* dl = b.dl + r0;
  const int* org = b.org + r0;
  const double* tau = b.tau + r0;
  const double dli = dl[i];
  double p = 1.0;
  for (int j = lane; j < k; j += 64)
    if (j != i) p *= ((dli - dl[org[j]]) - tau[j]) / (dli - dl[j]);
  p = wave_prod(p) * ((dli - dl[org[i]]) - tau[i]);
  if (lane == 0) {
    double z2 = -p;
    if (z2 < 0.0) z2 = 0.0;
    b.zh[r0 + i] = copysign(sqrt(z2), b.wv[r0 + i]);
  }
}

// --------------------------------------------- the first levels in one launch
// Rows [DC_LEAF b, ...) of the tridiagonal from 1 x 1 blocks to one block of
// at most DC_LEAF, everything in LDS, one workgroup per leaf. A level costs
// six launches when it runs on the whole matrix, whatever its size (60 us a
// level up to 64); here it costs six barriers, 96 us for the six levels
// against 370. Four lanes per root, per entry of zhat and per eigenvector; the
// merges' deflation passes by one wave together; their products on MFMA with
// the deflated columns as unit columns of V (blocks below 16 padded with
// zeros).
constexpr int DC_LEAF = 64;

struct DcLeaf {
  static constexpr int LD = DC_LEAF + 1;
  double Q[2][DC_LEAF * LD], V[DC_LEAF * LD];
  double D[2][DC_LEAF], ds[DC_LEAF], zs[DC_LEAF], dl[DC_LEAF], w[DC_LEAF], dval[DC_LEAF];
  double tau[DC_LEAF], zh[DC_LEAF], rcs[2 * DC_LEAF], rho[DC_LEAF], w2[DC_LEAF];
  int col[DC_LEAF], src[DC_LEAF], org[DC_LEAF], rcol[2 * DC_LEAF];
  int k[DC_LEAF], nrot[DC_LEAF];   // of the merge that starts at this row
};

// sum over the four lanes of a quad, the same bits in each
__device__ __forceinline__ double quad_sum(double v) {
  v += row_partner<1>(v);
  v += row_partner<2>(v);
  return v;
}

// The deflation pass of every merge of a level (aligned groups of s rows, s
// <= 64) by one wave, lane = sorted position. The rules are dc_deflate's: an
// entry with a negligible z is dropped, and consecutive kept entries that
// nearly coincide are rotated into one, which carries N = sum d z^2 and
// Z2 = sum z^2 of its run. Tests of neighbours with their own values find
// where a run starts; sums from that start on (a scan) give every later test
// of the run at once, and the first that fails ends it. One turn of the loop
// per run of two or more, against one step per entry (22 us for 64).
__device__ __forceinline__ void dc_leaf_deflate(DcLeaf& L, int lane, int s, int half, int nl) {
  const int r0 = lane / s * s, sm = min(s, nl - r0);
  const bool in = sm > half && lane < nl;
  const unsigned long long seg = (s == 64 ? ~0ull : ((1ull << s) - 1)) << r0;
  const unsigned long long below = (1ull << lane) - 1;
  const double d = in ? L.ds[lane] : 0.0, z = in ? L.zs[lane] : 0.0;
  const double rho = in ? L.rho[r0] : 0.0;
  double dm = fabs(d), zm = fabs(z);
  for (int o = 1; o < s; o <<= 1) {
    dm = fmax(dm, __shfl_xor(dm, o, 64));
    zm = fmax(zm, __shfl_xor(zm, o, 64));
  }
  const double tol = 8.0 * ITG_DC_EPS * fmax(dm, zm), tol2 = tol * tol;
  const bool kept = in && rho * fabs(z) > tol;
  const unsigned long long km = __ballot(kept) & seg;
  const double z2 = z * z;
  // the kept entry before this one (its lane; -1: none)
  const int pv = (km & below) ? 63 - __clzll(km & below) : -1;
  const double dp0 = __shfl(d, pv < 0 ? lane : pv, 64), zp0 = __shfl(z, pv < 0 ? lane : pv, 64);
  auto close = [&](double N, double Z2) {
    const double T2 = Z2 + z2, x = d * Z2 - N;
    return x * x * z2 <= tol2 * Z2 * T2 * T2;
  };
  const bool pair = kept && pv >= 0 && close(dp0 * (zp0 * zp0), zp0 * zp0);
  const unsigned long long pm = __ballot(pair) & seg;
  unsigned long long rot = 0;     // entries rotated onto (this group's)
  double N = d * z2, Z2 = z2;     // sums of the run up to this entry
  double Np = 0.0, Zp = 0.0;      // and before it
  int cur = r0;                   // entries up to here are settled
  while (true) {
    const unsigned long long m = cur >= 64 ? 0 : pm & (~0ull << cur) & ~(1ull << cur);
    // a start needs its predecessor at or after cur, which holds for any
    // kept entry after cur (cur itself is kept once a run has ended there)
    if (!__any(m != 0)) break;
    const bool have = m != 0;
    const int j0 = have ? __ffsll(m) - 1 : 0;
    const int s0 = have ? 63 - __clzll(km & ((1ull << j0) - 1)) : 0;
    double sn = have && kept && lane >= s0 ? d * z2 : 0.0;
    double sz = have && kept && lane >= s0 ? z2 : 0.0;
    for (int o = 1; o < s; o <<= 1) {
      const double un = __shfl_up(sn, o, 64), uz = __shfl_up(sz, o, 64);
      if (lane - r0 >= o) {
        sn += un;
        sz += uz;
      }
    }
    // the sums before this entry: those of the kept entry before it
    const double en = __shfl(sn, pv < 0 ? lane : pv, 64), ez = __shfl(sz, pv < 0 ? lane : pv, 64);
    const bool fail = have && kept && lane > s0 && !close(en, ez);
    const unsigned long long fm = __ballot(fail) & seg;
    if (have) {
      const int jf = fm ? __ffsll(fm) - 1 : r0 + s;   // first entry past the run
      const unsigned long long upto = jf >= 64 ? ~0ull : (1ull << jf) - 1;
      rot |= km & upto & ~((2ull << s0) - 1);
      if (kept && lane > s0 && lane < jf) {
        N = sn;
        Z2 = sz;
        Np = en;
        Zp = ez;
      }
      cur = jf;
    }
  }
  const bool myrot = (rot >> lane) & 1;
  // a kept entry survives unless the next kept one is rotated onto
  const unsigned long long later = km & ~below & ~(1ull << lane);
  const int nx = later ? __ffsll(later) - 1 : 64;
  const bool out = kept && !(nx < 64 && ((rot >> nx) & 1));
  const unsigned long long om = __ballot(out) & seg;
  const bool drop = in && !kept;
  const unsigned long long dm2 = __ballot(drop || myrot) & seg;
  const int col = in ? L.col[lane] : lane;
  const int pcol = __shfl(col, pv < 0 ? lane : pv, 64);
  const bool psingle = pv >= 0 && !((rot >> pv) & 1);   // a run of one before this entry
  const int k = __popcll(om);
  if (out) {
    const int q = r0 + __popcll(om & below);
    L.dl[q] = myrot ? N / Z2 : d;
    L.w[q] = myrot ? sqrt(Z2) : z;
    L.src[q] = col;
  }
  if (drop || myrot) {
    const int q = __popcll(dm2 & below);
    double v = d;
    if (myrot) {
      const double it = 1.0 / sqrt(Zp + z2);
      const double c = z * it, sg = -(psingle ? zp0 : sqrt(Zp)) * it;
      const double dp = psingle ? dp0 : Np / Zp;
      const int x = r0 + __popcll(rot & below);
      L.rcol[2 * x] = pcol;
      L.rcol[2 * x + 1] = col;
      L.rcs[2 * x] = c;
      L.rcs[2 * x + 1] = sg;
      v = dp * c * c + d * sg * sg;
    }
    L.dval[r0 + q] = v;
    L.src[r0 + k + q] = myrot ? pcol : col;
  }
  double w2 = out ? Z2 : 0.0;
  for (int o = 1; o < s; o <<= 1) w2 += __shfl_xor(w2, o, 64);
  if (in && lane == r0) {
    L.k[r0] = k;
    L.nrot[r0] = __popcll(rot);
    L.w2[r0] = w2;
  }
}

__global__ __launch_bounds__(256) void dc_leaf_kernel(int n, const double* __restrict__ d,
                                                      const double* __restrict__ e,
                                                      double* __restrict__ Qg,
                                                      double* __restrict__ Dg) {
  extern __shared__ __attribute__((aligned(16))) char dc_leaf_lds[];
  DcLeaf& L = *(DcLeaf*)dc_leaf_lds;
  constexpr int LD = DcLeaf::LD;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r00 = blockIdx.x * DC_LEAF, nl = min(DC_LEAF, n - r00);
  const int g = t >> 2, q4 = t & 3;   // row / root / column of four lanes
  for (int x = t; x < DC_LEAF * LD; x += 256) {
    L.Q[0][x] = x % LD == x / LD ? 1.0 : 0.0;
    L.Q[1][x] = 0.0;
  }
  if (t < DC_LEAF) {
    double v = 0.0;
    const int c = r00 + t;
    if (t < nl) {
      v = d[c];
      if (c > 0) v -= fabs(e[c - 1]);
      if (c < n - 1) v -= fabs(e[c]);
    }
    L.D[0][t] = v;
  }
  __syncthreads();
  int cur = 0;
  for (int half = 1; half < nl; half *= 2, cur ^= 1) {
    const int s = 2 * half;
    const int r0 = g / s * s, sm = min(s, nl - r0);   // this row's merge
    const bool act = sm > half;
    const int i = g - r0;
    double* Q = L.Q[cur];
    double* D = L.D[cur];
    // z and the position in the merge's ascending order (NaN after all
    // others, so that the positions are a permutation whatever D holds)
    if (act && g < nl) {
      int before = 0;
      const double dv = D[g], dg = fmin(dv, INFINITY);
      for (int c = q4; c < sm; c += 4) {
        const double dc = fmin(D[r0 + c], INFINITY);
        before += (dc < dg || (dc == dg && c < i)) ? 1 : 0;
      }
      before += __builtin_amdgcn_mov_dpp(before, 0xB1, 0xF, 0xF, false);
      before += __builtin_amdgcn_mov_dpp(before, 0x4E, 0xF, 0xF, false);
      if (q4 == 0) {
        const double beta = e[r00 + r0 + half - 1];
        const double sg = beta >= 0.0 ? 1.0 : -1.0;
        const double z = i < half ? Q[g * LD + r0 + half - 1] : sg * Q[g * LD + r0 + half];
        L.ds[r0 + before] = dv;
        L.zs[r0 + before] = z * 0.7071067811865476;
        L.col[r0 + before] = g;
        if (i == 0) L.rho[r0] = 2.0 * fabs(beta);
      }
    }
    __syncthreads();
    if (wave == 0) dc_leaf_deflate(L, lane, s, half, nl);
    __syncthreads();
    const int k = act ? L.k[r0] : 0;
    if (t < nl) {
      // the deflation's rotations, thread = row of Q
      const int b0 = t / s * s;
      if (min(s, nl - b0) > half) {
        const int nr = L.nrot[b0];
        for (int x = 0; x < nr; ++x) {
          const int pc = L.rcol[2 * b0 + 2 * x], qc = L.rcol[2 * b0 + 2 * x + 1];
          const double c = L.rcs[2 * b0 + 2 * x], sn = L.rcs[2 * b0 + 2 * x + 1];
          const double u = Q[pc * LD + t], v = Q[qc * LD + t];
          Q[pc * LD + t] = c * u + sn * v;
          Q[qc * LD + t] = c * v - sn * u;
        }
      }
    }
    const double* dl = L.dl + r0;
    const double* w = L.w + r0;
    if (act && i < k) {
      const double rho = L.rho[r0];
      auto ev = [&](int o, double tau, int side, double* dpo, double* dpf, double* absum) {
        double f = 0.0, po = 0.0, pf = 0.0, ab = 0.0;
        const double dlo = dl[o];
#pragma unroll 4
        for (int j = q4; j < k; j += 4) {
          const double del = (dl[j] - dlo) - tau;
          const double u = w[j] / del;
          const double term = rho * w[j] * u;
          f += term;
          ab += fabs(term);
          const double dt = rho * u * u;
          const bool origin_side = side > 0 ? (j <= o) : (j >= o);
          if (origin_side) po += dt; else pf += dt;
        }
        *dpo = quad_sum(po);
        *dpf = quad_sum(pf);
        *absum = 1.0 + quad_sum(ab);
        return 1.0 + quad_sum(f);
      };
      int o;
      double tv;
      dc_secular_root_with(i, k, dl, rho, L.w2[r0], ev, &o, &tv);
      if (q4 == 0) {
        L.org[g] = o;
        L.tau[g] = tv;
      }
    }
    __syncthreads();
    const int* org = L.org + r0;
    const double* tau = L.tau + r0;
    if (act && i < k) {
      // zhat_i (Gu-Eisenstat, as dc_zhat)
      const double dli = dl[i];
      double p = 1.0;
#pragma unroll 4
      for (int j = q4; j < k; j += 4)
        if (j != i) p *= ((dli - dl[org[j]]) - tau[j]) / (dli - dl[j]);
      p *= row_partner<1>(p);
      p *= row_partner<2>(p);
      p *= (dli - dl[org[i]]) - tau[i];
      if (q4 == 0) L.zh[g] = copysign(sqrt(p < 0.0 ? -p : 0.0), w[i]);
    }
    __syncthreads();
    {
      // column g of V: an eigenvector of the rank-one update, or a unit
      // column (deflated, or a block without a sibling at this level)
      const int S = s < 16 ? 16 : s, b0 = g / S * S;
      double lamo = 0.0, tj = 0.0, inv = 0.0;
      const bool root = act && g < nl && i < k;
      if (root) {
        lamo = dl[org[i]];
        tj = tau[i];
        double s2 = 0.0;
#pragma unroll 4
        for (int j = q4; j < k; j += 4) {
          const double v = L.zh[r0 + j] / ((dl[j] - lamo) - tj);
          s2 += v * v;
        }
        inv = 1.0 / sqrt(quad_sum(s2));
      }
#pragma unroll 4
      for (int x = b0 + q4; x < b0 + S; x += 4) {
        const int j = x - r0;
        double v;
        if (root) v = j >= 0 && j < k ? L.zh[x] / ((dl[j] - lamo) - tj) * inv : 0.0;
        else v = x == g ? 1.0 : 0.0;
        L.V[g * LD + x] = v;
      }
      if (q4 == 0) {
        L.D[cur ^ 1][g] = root ? lamo + tj : act && g < nl ? L.dval[r0 + i - k] : D[g];
        if (!act || g >= nl) L.src[g] = g;
      }
    }
    __syncthreads();
    {
      // Q' = Q(:, src) V, blocks of S on the diagonal
      const int S = s < 16 ? 16 : s, ts = S / 16;
      const int lr = lane & 15, lg = lane >> 4;
      for (int tile = wave; tile < DC_LEAF / S * ts * ts; tile += 4) {
        const int b0 = tile / (ts * ts) * S, in = tile % (ts * ts);
        const int row = b0 + in % ts * 16, cj = b0 + in / ts * 16;
        typedef double d4 __attribute__((ext_vector_type(4)));
        d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int x = b0; x < b0 + S; x += 4) {
          const double a = Q[L.src[x + lg] * LD + row + lr];
          const double b = L.V[(cj + lr) * LD + x + lg];
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) L.Q[cur ^ 1][(cj + lr) * LD + row + 4 * r + lg] = acc[r];
      }
    }
    __syncthreads();
  }
  for (int x = t; x < nl * nl; x += 256) {
    const int r = x % nl, c = x / nl;
    Qg[(size_t)(r00 + c) * n + r00 + r] = L.Q[cur][c * LD + r];
  }
  if (t < nl) Dg[r00 + t] = L.D[cur][t];
}

// column j of the rank-one eigenvector matrix, normalised (one wave per column)
__global__ __launch_bounds__(256) void dc_vec_kernel(int n, int s_lvl, int half, double* __restrict__ Vb,
                                                     DcBufs b) {
  int m = blockIdx.x, r0, s;
  if (!merge_range(n, s_lvl, half, m, r0, s)) return;
  int k = b.meta[3 * m];
  int lane = threadIdx.x & 63;
  int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (j >= k) return;
  const double* dl = b.dl + r0;
  double lamo = dl[b.org[r0 + j]];
  double tj = b.tau[r0 + j];
  double s2 = 0.0;
  for (int i = lane; i < k; i += 64) {
    double v = b.zh[r0 + i] / ((dl[i] - lamo) - tj);
    s2 += v * v;
  }
  for (int o = 32; o > 0; o >>= 1) s2 += __shfl_xor(s2, o, 64);
  double inv = 1.0 / sqrt(s2);
  double* Vm = Vb + (size_t)r0 * s_lvl;
  for (int i = lane; i < k; i += 64)
    Vm[i + (size_t)j * k] = b.zh[r0 + i] / ((dl[i] - lamo) - tj) * inv;
}

// new block columns: nondeflated (gemm part, small merges only), deflated
// copies, and eigenvalues
__global__ void dc_apply_kernel(int n, int s_lvl, int half, const double* __restrict__ Q,
                                double* __restrict__ Qn, const double* __restrict__ Vb,
                                double* __restrict__ Dn, DcBufs b, int do_gemm) {
  int m = blockIdx.x, r0, s;
  if (!merge_range(n, s_lvl, half, m, r0, s)) return;
  int k = b.meta[3 * m];
  int64_t tot = (int64_t)s * s;
  for (int64_t e = (int64_t)blockIdx.y * blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.y * blockDim.x) {
    int r = (int)(e % s), jc = (int)(e / s);
    if (jc < k) {
      if (r == 0) Dn[r0 + jc] = b.dl[r0 + b.org[r0 + jc]] + b.tau[r0 + jc];
      if (!do_gemm) continue;
      const double* Vm = Vb + (size_t)r0 * s_lvl + (size_t)jc * k;
      double acc = 0.0;
      for (int t = 0; t < k; ++t) acc += Q[(size_t)b.gcol[r0 + t] * n + r0 + r] * Vm[t];
      Qn[(size_t)(r0 + jc) * n + r0 + r] = acc;
    } else {
      int t2 = jc - k;
      if (r == 0) Dn[r0 + jc] = b.dval[r0 + t2];
      Qn[(size_t)(r0 + jc) * n + r0 + r] = Q[(size_t)b.dcol[r0 + t2] * n + r0 + r];
    }
  }
}

// a trailing block with no sibling at this level is carried over unchanged
__global__ void dc_carry_kernel(int n, int r0, int s, const double* __restrict__ Q,
                                double* __restrict__ Qn, const double* __restrict__ D,
                                double* __restrict__ Dn) {
  int64_t tot = (int64_t)s * s;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int r = (int)(e % s), c = (int)(e / s);
    Qn[(size_t)(r0 + c) * n + r0 + r] = Q[(size_t)(r0 + c) * n + r0 + r];
    if (r == 0) Dn[r0 + c] = D[r0 + c];
  }
}

__global__ void dc_table_kernel(int k, const int* __restrict__ gcol, int n, int64_t* __restrict__ tab) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < k) tab[t] = (int64_t)gcol[t] * n;
}

__global__ __launch_bounds__(1024) void dc_final_sort_kernel(int n, const double* __restrict__ D,
                                                             int* __restrict__ perm,
                                                             double* __restrict__ wout) {
  extern __shared__ double lds_d[];
  int np2 = 1;
  while (np2 < n) np2 <<= 1;
  double* key = lds_d;
  int* val = (int*)(key + np2);
  for (int i = threadIdx.x; i < np2; i += blockDim.x) {
    key[i] = i < n ? -D[i] : INFINITY;
    val[i] = i < n ? i : 0;
  }
  __syncthreads();
  bitonic_sort(key, val, np2);
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    perm[i] = val[i];
    wout[i] = -key[i];
  }
}

// out = min over p < k of perm[p] among those < kt (else kt), as a double
__global__ __launch_bounds__(256) void dc_first_kept_kernel(const int* __restrict__ perm, int k,
                                                            int kt, double* __restrict__ out) {
  __shared__ int sh[4];
  int v = kt;
  for (int p = threadIdx.x; p < k; p += 256) v = min(v, perm[p] < kt ? perm[p] : kt);
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = (double)min(min(sh[0], sh[1]), min(sh[2], sh[3]));
}

__global__ void gather_cols_kernel(int n, int k, const double* __restrict__ Q,
                                   const int* __restrict__ perm, double* __restrict__ U) {
  int64_t tot = (int64_t)n * k;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int r = (int)(e % n), c = (int)(e / n);
    U[e] = Q[(size_t)perm[c] * n + r];
  }
}

struct Carver {
  char* base;
  size_t off = 0;
  template <typename T>
  T* take(size_t count) {
    off = (off + 255) & ~(size_t)255;
    T* p = (T*)(base + off);
    off += count * sizeof(T);
    return p;
  }
};

int set_lds_limit(itg_ctx* ctx) {
  if (ctx->lds_set & ITG_LDS_EIGH) return ITG_OK;
  ITG_HIP(ctx, hipFuncSetAttribute((const void*)dc_prepare_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, DC_ZLDS * 28));
  ITG_HIP(ctx, hipFuncSetAttribute((const void*)trd_mid_kernel<7, 10, 4>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, MID_LDS));
  ITG_HIP(ctx, hipFuncSetAttribute((const void*)dc_leaf_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(DcLeaf)));
  ITG_HIP(ctx, hipFuncSetAttribute((const void*)dc_final_sort_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 8192 * 12));
  ctx->lds_set |= ITG_LDS_EIGH;
  return ITG_OK;
}

}  // namespace

static int eig_workspace(itg_ctx* ctx, size_t bytes, void** out) {
  if (bytes > ctx->eig_ws_bytes) {
    if (ctx->eig_ws) {
      ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
      ITG_HIP(ctx, hipFree(ctx->eig_ws));
      ctx->eig_ws = nullptr;
      ctx->eig_ws_bytes = 0;
    }
    if (hipMalloc(&ctx->eig_ws, bytes) != hipSuccess) {
      hipGetLastError();
      return itg_fail(ctx, ITG_EOOM, "eigensolver workspace of %zu bytes failed", bytes);
    }
    ctx->eig_ws_bytes = bytes;
  }
  *out = ctx->eig_ws;
  return ITG_OK;
}

// From this many trailing rows on: the copy, the loads and the read-back cost
// 31 us, a column of the chip-wide kernels 5 us more than one of these (n = 220
// whole: 1045 us without, 934 with; even at six columns). Up to MID_MAX rows:
// the registers and LDS of 256 CUs hold no more.
constexpr int MID_MIN = TRD_TAIL + 8;
constexpr int MID_SKIP = 32;

// Columns p .. n - TRD_TAIL - 1 by the resident kernels, the trailing block
// handed from one to the next as it shrinks; *ok = false if a wait ran out
// (A as before the call).
static int trd_resident(itg_ctx* ctx, int n, int p, double* A, double* d, double* e, double* tau,
                        double* copy, mid_t* ring, bool* ok) {
  static std::mutex turn[64];   // one reduction at a time on a device
  const char* env = getenv("ITG_TRD_WAIT_MS");
  const long long limit = (env ? atoll(env) : 50) * 100000LL;
  int dev = 0;
  ITG_HIP(ctx, hipGetDevice(&dev));
  int* stop = (int*)(ring + 4 * 2 * MID_MAX);
  hipStream_t st = ctx->stream;
  const int m0 = n - p, p0 = p;
  trd_copy_kernel<<<itg_blocks((int64_t)m0 * m0, 256, 8192), 256, 0, st>>>(A, n, p, copy, false);
  int stopped = 0;
  // no other context waits for what this stream still has queued
  if (itg_live_contexts(dev) > 1) ITG_HIP(ctx, hipStreamSynchronize(st));
  {
    std::lock_guard<std::mutex> lock(turn[dev & 63]);
    for (int end; p < n - TRD_TAIL; p = end) {
      const int m = n - p, K = (m + 511) / 512;
      end = K == 1 ? n - TRD_TAIL : n - 512 * (K - 1);
      const int count = 4 * 2 * 512 * K;
      trd_mid_clear_kernel<<<(count + 255) / 256, 256, 0, st>>>(ring, count, stop, p == p0);
      auto go = [&](auto kernel, int rows, size_t lds) {
        kernel<<<(m + rows - 1) / rows, 512, lds, st>>>(A, n, p, end - p, d, e, tau, ring, stop,
                                                        limit);
      };
      if (K == 1) go(trd_mid_kernel<1, 16, 0>, 16, 0);
      else if (K == 2) go(trd_mid_kernel<2, 16, 0>, 16, 0);
      else if (K == 3) go(trd_mid_kernel<3, 16, 0>, 16, 0);
      else if (K == 4) go(trd_mid_kernel<4, 16, 0>, 16, 0);
      else if (K == 5) go(trd_mid_kernel<5, 16, 0>, 16, 0);
      else if (K == 6) go(trd_mid_kernel<6, 12, 0>, 12, 0);
      else go(trd_mid_kernel<7, 10, 4>, 14, MID_LDS);
      ITG_LAUNCH_CHECK(ctx);
    }
    ITG_HIP(ctx, hipMemcpyAsync(&stopped, stop, sizeof(int), hipMemcpyDeviceToHost, st));
    ITG_HIP(ctx, hipStreamSynchronize(st));
  }
  *ok = stopped == 0;
  // a device that is shared for long: from the second run-out in a row on,
  // 2, 4, .. MID_SKIP calls of this context do without before the next try,
  // so that the waits cost them at most limit / MID_SKIP each
  ctx->trd_outs = stopped ? std::min(ctx->trd_outs + 1, 31) : 0;
  ctx->trd_skip = ctx->trd_outs > 1 ? std::min(1 << (ctx->trd_outs - 1), MID_SKIP) : 0;
  if (stopped) {
    trd_copy_kernel<<<itg_blocks((int64_t)m0 * m0, 256, 8192), 256, 0, st>>>(A, n, p0, copy, true);
    ITG_LAUNCH_CHECK(ctx);
  }
  return ITG_OK;
}

// Tridiagonalise A (n x n FP64, full symmetric storage) in place: d, e out;
// reflectors left in A's strictly lower part (v_j(j+1) = 1 explicit), tau out.
static int tridiagonalize(itg_ctx* ctx, int n, double* A, double* d, double* e, double* tau,
                          double* VW, double* Ypart, double* ab, double* pnorm, double* pyv,
                          double* sc, double* copy, double* ring) {
  // VW = [V | W | V], n x NB each: the trailing update of a full panel is one
  // K = 2 NB product A22 -= [V W] [W V]^T
  double* Vp = VW;
  double* Wp = VW + (size_t)n * NB;
  double* V2 = VW + 2 * (size_t)n * NB;
  bool resident = copy != nullptr;
  for (int p = 0, nbp; p < n; p += nbp) {
    if (resident && n - p <= MID_MAX && n - p >= MID_MIN && ctx->trd_skip > 0) {
      --ctx->trd_skip;
      resident = false;
    }
    if (resident && n - p <= MID_MAX && n - p >= MID_MIN) {
      int rc = trd_resident(ctx, n, p, A, d, e, tau, copy, (mid_t*)ring, &resident);
      if (rc) return rc;
      if (resident) p = n - TRD_TAIL;
      resident = false;
    }
    if (n - p <= TRD_TAIL) {
      // every earlier panel's update is applied: the rest in one block
      const int m = n - p;
      if (m > 128) {
        trd_tail_kernel<6><<<1, 512, 0, ctx->stream>>>(A, n, p, d, e, tau);
      } else if (m > 64) {
        trd_tail_kernel<4><<<1, 512, 0, ctx->stream>>>(A, n, p, d, e, tau);
      } else if (m >= 2) {
        trd_tail_kernel<2><<<1, 512, 0, ctx->stream>>>(A, n, p, d, e, tau);
      } else {
        trd_last_kernel<<<1, 1, 0, ctx->stream>>>(A, n, d, tau);
      }
      ITG_LAUNCH_CHECK(ctx);
      return ITG_OK;
    }
    // the last panel stops where the tail kernel can take over
    nbp = std::min(NB, n - TRD_TAIL - p);
    const int npn = (n + TRD_ROWS - 1) / TRD_ROWS;
    int pn_off = 0, pn_cnt = npn;
    if (p < n - 1) {
      trd_colnorm_kernel<<<npn, 256, 0, ctx->stream>>>(A, n, p, pnorm);
      ITG_LAUNCH_CHECK(ctx);
    }
    for (int i = 0; i < nbp; ++i) {
      int j = p + i;
      if (j == n - 1) {
        trd_last_kernel<<<1, 1, 0, ctx->stream>>>(A, n, d, tau);
        ITG_LAUNCH_CHECK(ctx);
        break;
      }
      int m = n - j - 1;
      int T = (m + TS - 1) / TS;
      int ntiles = T * (T + 1) / 2;
      itg_tev tk = itg_tevents(ctx, ITG_K_TRD_SYMV);
      hipExtLaunchKernelGGL(trd_symv_kernel, dim3((ntiles + 7) / 8 * 8 + (i + 7) / 8 * 8), dim3(256),
                            0, ctx->stream,
                            tk.a, tk.b, 0, (const double*)A, n, j, i,
                            (const double*)(pnorm + pn_off), pn_cnt, Vp, (const double*)Wp, V2,
                            Ypart, ab, pyv, ntiles, d, e, tau, sc);
      ITG_LAUNCH_CHECK(ctx);
      // lower triangle of A22 read once, the panel pairs over m rows
      itg_tcommit(ctx, tk, ITG_K_TRD_SYMV, 2.0 * m * (m + 2.0 * i),
                  8.0 * (0.5 * m * (m + TS) + 2.0 * i * m + 2.0 * T * m));
      int next = (i + 1 < nbp) ? 1 : 0;
      const int b0 = (j + 1) / POST_ROWS;
      const int nblk = (n + POST_ROWS - 1) / POST_ROWS - b0;
      itg_tev tp = itg_tevents(ctx, ITG_K_TRD_POST);
      hipExtLaunchKernelGGL(trd_post_kernel, dim3(nblk), dim3(256), 0, ctx->stream, tp.a, tp.b, 0,
                            A, n, j, i, ntiles, (const double*)Vp, Wp, (const double*)Ypart, T,
                            (const double*)ab, (const double*)pyv, (const double*)tau,
                            (const double*)e, (const double*)sc, next, pnorm, b0);
      ITG_LAUNCH_CHECK(ctx);
      // the next column's reflector norm: partials of these blocks only
      pn_off = b0;
      pn_cnt = nblk;
      itg_tcommit(ctx, tp, ITG_K_TRD_POST, 8.0 * m * (i + 1), 8.0 * m * (2.0 * i + 5 + T));
    }
    int q = p + nbp;
    if (q < n) {
      int m2 = n - q;
      double* A22 = A + (size_t)q * n + q;
      int rc;
      // the tiled symv reads A22's 64 x 64 tiles on and below its diagonal
      // (diagonal tiles whole), the post kernel and the column norms the
      // lower part: the lower triangle plus one 128-tile band suffices
      if (nbp == NB) {
        rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'T', m2, m2, 2 * NB, -1.0,
                               Vp + q, n, Wp + q, n, 1.0, A22, n, true);
        if (rc) return rc;
      } else {
        rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'T', m2, m2, nbp, -1.0, Vp + q,
                               n, Wp + q, n, 1.0, A22, n, true);
        if (rc) return rc;
        rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'T', m2, m2, nbp, -1.0, Wp + q,
                               n, Vp + q, n, 1.0, A22, n, true);
        if (rc) return rc;
      }
    }
  }
  return ITG_OK;
}

// Eigen-decomposition of the tridiagonal (d, e): eigenvalues D (unsorted)
// and eigenvectors as the columns of the returned buffer (Qa or Qb).
// With `top` non-null the last merge's eigenvector product is not launched
// but returned in *top (top->M = 0 if there is none), for the caller to run
// on the columns it keeps.
static int tridiag_dc(itg_ctx* ctx, int n, const double* d, const double* e, double* Qa,
                      double* Qb, double* Da, double* Db, double* Vb, DcBufs bufs, int64_t* tab,
                      double** Qout, double** Dout, GettArgs* top) {
  if (top) top->M = 0;
  dc_init_kernel<<<itg_blocks((int64_t)n * n, 256, 16384), 256, 0, ctx->stream>>>(n, Qa, Qb);
  dc_leaf_kernel<<<(n + DC_LEAF - 1) / DC_LEAF, 256, sizeof(DcLeaf), ctx->stream>>>(n, d, e, Qa, Da);
  ITG_LAUNCH_CHECK(ctx);
  double *Q = Qa, *Qn = Qb, *D = Da, *Dn = Db;
  std::vector<int> meta;
  for (int half = DC_LEAF; half < n; half *= 2) {
    int s_lvl = 2 * half;
    int nm = (n + s_lvl - 1) / s_lvl;
    size_t lds = (size_t)s_lvl * (sizeof(double) + sizeof(int) +
                                  (s_lvl <= DC_ZLDS ? sizeof(double) + 2 * sizeof(int) : 0));
    dc_prepare_kernel<<<nm, 1024, lds, ctx->stream>>>(n, s_lvl, half, D, Q, e, bufs);
    ITG_LAUNCH_CHECK(ctx);
    // the host needs the merges' sizes only to launch their products
    const bool small = s_lvl <= SMALL_MERGE;
    if (!small) {
      meta.assign(3 * nm, 0);
      ITG_HIP(ctx, hipMemcpyAsync(meta.data(), bufs.meta, 3 * nm * sizeof(int),
                                  hipMemcpyDeviceToHost, ctx->stream));
      ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    dim3 g256(nm, (s_lvl + 255) / 256);
    dc_rotate_kernel<<<g256, 256, 0, ctx->stream>>>(n, s_lvl, half, Q, bufs);
    dim3 g4(nm, (s_lvl + 3) / 4);
    dc_secular_kernel<<<g4, 256, 0, ctx->stream>>>(n, s_lvl, half, bufs);
    dc_zhat_kernel<<<g4, 256, 0, ctx->stream>>>(n, s_lvl, half, bufs);
    dc_vec_kernel<<<dim3(nm, (s_lvl + 3) / 4), 256, 0, ctx->stream>>>(n, s_lvl, half, Vb, bufs);
    ITG_LAUNCH_CHECK(ctx);
    if (!small) {
      for (int m = 0; m < nm; ++m) {
        int r0 = m * s_lvl, s = std::min(s_lvl, n - r0), k = meta[3 * m];
        if (s <= half || k == 0) continue;
        dc_table_kernel<<<(k + 255) / 256, 256, 0, ctx->stream>>>(k, bufs.gcol + r0, n, tab);
        // Qn[r0.., r0+j] (j < k) = sum_t Q[r0.., gcol[t]] V[t, j], computed as
        // C^T(j, r) = V^T(j, t) A^T(t, r) so the stores run along rows
        GettArgs g = {};
        g.A = Vb + (size_t)r0 * s_lvl;
        g.B = Q + r0;
        g.C = Qn + (size_t)r0 * n + r0;
        g.M = k; g.N = s; g.K = k;
        g.sAm = k; g.sAk = 1;
        g.sBk = -1; g.tBk = tab; g.sBn = 1;
        g.sCm = n; g.sCn = 1;
        g.alpha = 1.0; g.beta = 0.0;
        if (top && s_lvl >= n) {
          *top = g;   // the last merge (nm == 1, r0 == 0)
          continue;
        }
        int rc = itg_gett_launch(ctx, ITG_F64, ITG_MODE_NATIVE, &g, true, false);
        if (rc) return rc;
      }
    }
    dim3 gap(nm, (unsigned)std::min<int64_t>(((int64_t)s_lvl * s_lvl + 255) / 256, 8192));
    dc_apply_kernel<<<gap, 256, 0, ctx->stream>>>(n, s_lvl, half, Q, Qn, Vb, Dn, bufs, small ? 1 : 0);
    ITG_LAUNCH_CHECK(ctx);
    int r0l = (nm - 1) * s_lvl, sl = n - r0l;
    if (sl <= half) {
      dc_carry_kernel<<<itg_blocks((int64_t)sl * sl, 256, 4096), 256, 0, ctx->stream>>>(n, r0l, sl, Q, Qn, D, Dn);
      ITG_LAUNCH_CHECK(ctx);
    }
    std::swap(Q, Qn);
    std::swap(D, Dn);
  }
  *Qout = Q;
  *Dout = D;
  return ITG_OK;
}

// U (m x k) <- H_0 ... H_{nrefl-1} U, reflector j in column j of A (leading
// dimension m) from row j + off on, v(j + off) = 1 stored and zeros above
// within its group. Groups of BT_GROUP reflectors go last to first: Y = V^T U,
// G = V^T V, the group solve for X, U -= V X. `eye`: U is the identity's first
// k = nrefl columns (columns before a group's first are still untouched).
static int back_transform_groups(itg_ctx* ctx, int m, int nrefl, int off, int k, const double* A,
                                 const double* tau, double* U, bool eye, double* Y, double* X2,
                                 double* Gg) {
  if (nrefl < 1 || k < 1) return ITG_OK;
  for (int p0 = (nrefl - 1) / BT_GROUP * BT_GROUP; p0 >= 0; p0 -= BT_GROUP) {
    const int nbg = std::min(BT_GROUP, nrefl - p0);
    const int m2 = m - p0 - off, c0 = eye ? p0 : 0, kc = k - c0;
    const double* VG = A + (size_t)p0 * m + (p0 + off);   // rows p0+off.., columns p0..p0+nbg
    double* UG = U + (size_t)c0 * m + (p0 + off);
    int rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', nbg, kc, m2, 1.0, VG, m, UG,
                               m, 0.0, Y, nbg);
    if (rc) return rc;
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', nbg, nbg, m2, 1.0, VG, m, VG,
                           m, 0.0, Gg, nbg);
    if (rc) return rc;
    bt_group_solve_kernel<<<(kc + 15) / 16, 256, 0, ctx->stream>>>(nbg, kc, Y, Gg, tau + p0, X2);
    ITG_LAUNCH_CHECK(ctx);
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', m2, kc, nbg, -1.0, VG, m, X2,
                           nbg, 1.0, UG, m);
    if (rc) return rc;
  }
  return ITG_OK;
}

extern "C" int itg_eigh_trunc(itg_ctx* ctx, int dtype, int64_t n64, void* Ain, double* w,
                              void* Uout, int64_t maxdim, double cutoff, int abs_cut, int rel_cut,
                              int64_t* kout, double* truncerr, double* docut) {
  ITG_CHECK_CTX(ctx);
  const bool cplx = dtype == ITG_C64;   // Hermitian (heevd's route)
  if (!cplx) ITG_CHECK_DTYPE(ctx, dtype);
  if (n64 < 0) return itg_fail(ctx, ITG_EDIM, "eigh: negative dimension");
  if (n64 > 8192) return itg_fail(ctx, ITG_EUNSUPPORTED, "eigh: n = %lld > 8192", (long long)n64);
  if (!kout) return itg_fail(ctx, ITG_EARG, "eigh: null k");
  if (n64 == 0) {
    *kout = 0;
    if (truncerr) *truncerr = 0.0;
    if (docut) *docut = 0.0;
    return ITG_OK;
  }
  int rc = set_lds_limit(ctx);
  if (rc) return rc;
  int n = (int)n64;
  size_t nn = (size_t)n * n;
  bool f32 = dtype == ITG_F32;
  // the two-stage reduction (dense -> band -> tridiagonal) on request
  // (ITG_EIGH_TWOSTAGE=1, read per call): correct, but at n = 4096 it takes
  // 113 ms against 36 with the one-stage reduction, its bulge chasing and
  // tall-panel QRs being latency-bound
  const char* two_env = getenv("ITG_EIGH_TWOSTAGE");
  const bool two = !cplx && n >= TWO_STAGE_MIN && two_env && two_env[0] == '1';
  const size_t Tw = (size_t)(n + 63) / 64;   // tile rows of the tiled symv
  size_t bytes = (3 * nn + (f32 ? 2 * nn : 0)) * sizeof(double) + 3 * (size_t)n * NB * 8 +
                 (2 * (size_t)BT_GROUP * n + (size_t)BT_GROUP * BT_GROUP) * 8 +
                 (size_t)n * 8 * 25 + 4 * (size_t)n * NB * 8 + 64 * 1024 +
                 (Tw * n + Tw * (Tw + 1) / 2 + 64) * 8 + 64 * 256 +
                 ((size_t)n / POST_ROWS + 1) * 8 +
                 (two ? eig2::doubles_needed(n) * 8 + 256 : 0) +
                 (cplx ? (nn + itg_zhetrd_scratch_doubles(n) + 2 * (size_t)n) * 8 + 512 : 0);
  void* ws;
  rc = eig_workspace(ctx, bytes, &ws);
  if (rc) return rc;
  Carver cv{(char*)ws};
  double* Qa = cv.take<double>(nn);
  double* Qb = cv.take<double>(nn);
  double* Vbuf = cv.take<double>(nn);   // D&C merge vectors
  // complex: A stays the caller's (complex) matrix, U a real n x k staging
  // buffer for the tridiagonal's eigenvectors
  double* A = f32 ? cv.take<double>(nn) : cplx ? nullptr : (double*)Ain;
  double* U = (f32 || cplx) ? cv.take<double>(nn) : (double*)Uout;
  double* zscr = cplx ? cv.take<double>(itg_zhetrd_scratch_doubles(n)) : nullptr;
  double* ztau = cplx ? cv.take<double>(2 * (size_t)n) : nullptr;
  const size_t Tmax = (size_t)(n + TS - 1) / TS;
  double* VW = cv.take<double>(3 * (size_t)n * NB);
  double* Ypart = cv.take<double>(Tmax * n);
  double* ab = cv.take<double>(2 * NB);
  double* pnorm = cv.take<double>((size_t)n / POST_ROWS + 1);
  double* pyv = cv.take<double>(Tmax * (Tmax + 1) / 2 + 64);
  double* trd_sc = cv.take<double>(2);
  double* d = cv.take<double>(n);
  double* e = cv.take<double>(n);
  double* tau = cv.take<double>(n);
  double* Da = cv.take<double>(n);
  double* Db = cv.take<double>(n);
  DcBufs b;
  b.zs = cv.take<double>(n); b.dl = cv.take<double>(n);
  b.wv = cv.take<double>(n); b.dval = cv.take<double>(n); b.rcs = cv.take<double>(2 * (size_t)n);
  b.tau = cv.take<double>(n); b.zh = cv.take<double>(n); b.mrho = cv.take<double>(2 * (size_t)n);
  b.gcol = cv.take<int>(n); b.dcol = cv.take<int>(n);
  b.rcol = cv.take<int>(2 * (size_t)n); b.org = cv.take<int>(n); b.meta = cv.take<int>(3 * (size_t)n);
  int* perm = cv.take<int>(n);
  int64_t* tab = cv.take<int64_t>(n);
  double* Ygrp = cv.take<double>((size_t)BT_GROUP * n);
  double* X2grp = cv.take<double>((size_t)BT_GROUP * n);
  double* Ggrp = cv.take<double>((size_t)BT_GROUP * BT_GROUP);
  double* out3 = cv.take<double>(4);
  eig2::Bufs eb{};
  if (two) eig2::carve(n, cv.take<double>(eig2::doubles_needed(n)), &eb);
  if (cv.off > bytes) return itg_fail(ctx, ITG_EOOM, "eigh: workspace layout overflow");
  if (f32) {
    rc = itg_convert(ctx, (int64_t)nn, ITG_F32, Ain, ITG_F64, A);
    if (rc) return rc;
  }
  // 1. tridiagonalise
  if (cplx) rc = itg_zhetrd(ctx, n, Ain, d, e, ztau, zscr);
  else if (two) rc = eig2::reduce(ctx, n, A, d, e, eb);
  else {
    // the resident reduction reads its outcome back: not under capture, and
    // with every CU its workgroups need
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    ITG_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cap));
    const bool resident = cap == hipStreamCaptureStatusNone && ctx->num_cu >= MID_MAX / 14;
    rc = tridiagonalize(ctx, n, A, d, e, tau, VW, Ypart, ab, pnorm, pyv, trd_sc,
                        resident ? Qa : nullptr, Qb);
  }
  if (rc) return rc;
  // 2. divide and conquer
  double *Q, *D;
  GettArgs top = {};
  rc = tridiag_dc(ctx, n, d, e, Qa, Qb, Da, Db, Vbuf, b, tab, &Q, &D, &top);
  if (rc) return rc;
  // 3. sort descending, truncate
  {
    int np2 = 1;
    while (np2 < n) np2 <<= 1;
    dc_final_sort_kernel<<<1, 1024, (size_t)np2 * 12, ctx->stream>>>(n, D, perm, w);
    ITG_LAUNCH_CHECK(ctx);
  }
  int64_t k = n;
  double te = 0.0, dc = 0.0;
  if (cutoff >= 0.0 || (maxdim > 0 && maxdim < n)) {
    rc = itg_truncate_device_async(ctx, w, n, maxdim, 1, cutoff < 0.0 ? 0.0 : cutoff, abs_cut,
                                   rel_cut, ITG_TRUNC_NDTENSORS, out3);
    if (rc) return rc;
    double h[3];
    ITG_HIP(ctx, hipMemcpyAsync(h, out3, 3 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    k = (int64_t)h[0];
    te = h[1];
    dc = h[2];
  }
  // the last merge's eigenvector product, for its non-deflated columns from
  // the first one kept on (Q columns [0, top.M) are the non-deflated ones;
  // their eigenvalues increase with the column, so the kept ones are a tail)
  if (top.M > 0) {
    int64_t j0 = 0;
    if (k < n) {
      dc_first_kept_kernel<<<1, 256, 0, ctx->stream>>>(perm, (int)k, (int)top.M, out3 + 3);
      ITG_LAUNCH_CHECK(ctx);
      double h0;
      ITG_HIP(ctx, hipMemcpyAsync(&h0, out3 + 3, sizeof(double), hipMemcpyDeviceToHost,
                                  ctx->stream));
      ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
      j0 = (int64_t)h0;
    }
    if (j0 < top.M) {
      GettArgs g = top;
      g.A = (const double*)top.A + (size_t)j0 * top.sAm;
      g.C = (double*)top.C + (size_t)j0 * top.sCm;
      g.M = top.M - j0;
      rc = itg_gett_launch(ctx, ITG_F64, ITG_MODE_NATIVE, &g, true, false);
      if (rc) return rc;
    }
  }
  // 4. kept eigenvectors: gather, back-transform
  gather_cols_kernel<<<itg_blocks((int64_t)n * k, 256, 16384), 256, 0, ctx->stream>>>(n, (int)k, Q, perm, U);
  ITG_LAUNCH_CHECK(ctx);
  if (cplx) {
    rc = itg_zunmtr(ctx, n, (int)k, Ain, ztau, U, Uout);
  } else if (two) {
    rc = eig2::apply_q2(ctx, n, (int)k, U, eb);
    if (rc) return rc;
    static_assert(eig2::SB == NB, "panels of one width");
    bt_tau_kernel<<<(n + 255) / 256, 256, 0, ctx->stream>>>(eb.Tall, n - eig2::SB, tau);
    ITG_LAUNCH_CHECK(ctx);
    rc = back_transform_groups(ctx, n, n - eig2::SB, eig2::SB, (int)k, A, tau, U, false, Ygrp,
                               X2grp, Ggrp);
  } else {
    bt_clear_upper_kernel<<<itg_blocks((int64_t)n * n, 256, 16384), 256, 0, ctx->stream>>>(A, n);
    ITG_LAUNCH_CHECK(ctx);
    rc = back_transform_groups(ctx, n, n - 1, 1, (int)k, A, tau, U, false, Ygrp, X2grp, Ggrp);
  }
  if (rc) return rc;
  if (f32) {
    rc = itg_convert(ctx, (int64_t)n * k, ITG_F64, U, ITG_F32, Uout);
    if (rc) return rc;
  }
  *kout = k;
  if (truncerr) *truncerr = te;
  if (docut) *docut = dc;
  return ITG_OK;
}

// ====================================================================== QR
// Householder QR (culinearalgebra.jl:110-121): reflectors of W = A column by
// column, then Q = H_0...H_{r-1} [I; 0] by the same compact-WY
// back-transform, R = triu(W). Q of 2000 x 1000 in groups of 128 reflectors
// takes 0.45 ms; panel by panel (16 reflectors, two launches each), 1.45.
namespace {

// A reflector whose tail x below the pivot alpha has |x|^2 < QR_TINY2: near
// underflow, in its squares and in its products with other columns as small.
// Beside a pivot of QR_TINY_PIVOT or more the tail is less than 2^-60 of the
// column and counts as zero; else the reflector is formed from QR_UP times the
// tail (or QR_UP^2 times, if that is still as small), so that a matrix of any
// scale satisfies A = QR relative to itself. In the panel kernels that is the
// column's step taken again, which costs other matrices nothing to 1.5% (us,
// without and with: 2000 x 1000 3148 / 3150, 600 x 500 1205 / 1218, 3600 x 1500
// 8670 / 8795, 5000 x 600 6025 / 5848); as code of its own it cost 4.5%.
constexpr double QR_TINY2 = 0x1p-600, QR_TINY_PIVOT = 0x1p-240, QR_UP = 0x1p500;

__global__ __launch_bounds__(1024) void qr_reflect_kernel(double* __restrict__ W, int m, int j,
                                                          double* __restrict__ tau) {
  __shared__ double red[16];
  __shared__ double sc;
  double* a = W + (size_t)j * m;
  double xn2, up = 1.0;
  while (true) {
    double part = 0.0;
    for (int r = j + 1 + threadIdx.x; r < m; r += blockDim.x) part += (a[r] * up) * (a[r] * up);
    xn2 = block_sum(part, red);
    // the same in the whole workgroup
    if (!(xn2 < QR_TINY2) || !(fabs(a[j]) * up < QR_TINY_PIVOT) || up > QR_UP) break;
    up *= QR_UP;
  }
  __syncthreads();   // a[j] is read above
  if (threadIdx.x == 0) {
    const double alpha = a[j], au = alpha * up;
    double beta = alpha, tv = 0.0, scale = 0.0;
    if (!(xn2 < QR_TINY2) || (up > 1.0 && xn2 > 0.0)) {
      const double bu = -copysign(sqrt(au * au + xn2), au);
      beta = bu / up;
      tv = (bu - au) / bu;
      scale = 1.0 / (au - bu);
    }
    a[j] = beta;
    tau[j] = tv;
    sc = scale;
  }
  __syncthreads();
  double scale = sc;
  for (int r = j + 1 + threadIdx.x; r < m; r += blockDim.x) a[r] = a[r] * up * scale;
}

// W[j:m, c] -= tau_j v (v^T W[j:m, c]) for j < c < nend (the rest of the
// panel), one 256-thread block per column
__global__ __launch_bounds__(256) void qr_apply_kernel(double* __restrict__ W, int m, int nend,
                                                       int j, const double* __restrict__ tau) {
  __shared__ double sh4[4];
  const int c = j + 1 + blockIdx.x;
  if (c >= nend) return;
  const double tj = tau[j];
  if (tj == 0.0) return;
  const double* v = W + (size_t)j * m;
  double* col = W + (size_t)c * m;
  double s = 0.0;
  for (int r = j + threadIdx.x; r < m; r += 256) s += (r == j ? 1.0 : v[r]) * col[r];
  s = block_sum256(s, sh4);
  const double f = tj * s;
  for (int r = j + threadIdx.x; r < m; r += 256) col[r] -= f * (r == j ? 1.0 : v[r]);
}

// ------------------------------------------ QR of up to 8192 rows (blocked)
// Panels of QW columns: one workgroup factors the panel in registers, then
// the columns to the right take its block reflector in two launches.
constexpr int QW = 16;
constexpr int QR_MAX_ROWS = 8192;   // 16 rows a thread, 4 columns at a time
typedef double d4v_t __attribute__((ext_vector_type(4)));

// a double of lane l (wave-uniform l), in scalar registers
__device__ __forceinline__ double read_lane(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// element (l, c) of the panel's V, unit lower trapezoidal with w columns and
// m2 rows: the load is unconditional (clamped), so that a loop's loads all go
// out before any is used
__device__ __forceinline__ double qr_v(const double* __restrict__ A, int ld, int m2, int w, int l,
                                       int c) {
  const double v = A[min(l, m2 - 1) + (size_t)min(c, w - 1) * ld];
  return (l >= m2 || c >= w || l < c) ? 0.0 : (l == c ? 1.0 : v);
}

// element (l, c) of C (m2 x nc), zero outside
__device__ __forceinline__ double qr_c(const double* __restrict__ C, int ld, int m2, int nc, int l,
                                       int c) {
  const double v = C[min(l, m2 - 1) + (size_t)min(c, nc - 1) * ld];
  return (l >= m2 || c >= nc) ? 0.0 : v;
}

// Y = V^T C (QW x 16) over the 64 rows from b on, for one wave: a lane takes
// four consecutive rows of one column of each operand and spends them on four
// products; the 32 loads of the four row blocks go out together
template <typename F>
__device__ __forceinline__ d4v_t qr_vt_c(const double* __restrict__ A, int ld, int m2, int w,
                                         int b, int lr, int lg, d4v_t acc, F&& cel) {
  double va[4][4], vb[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int l = b + 16 * u + 4 * lg + q;
      va[u][q] = qr_v(A, ld, m2, w, l, lr);
      vb[u][q] = cel(l, lr);
    }
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u][q], vb[u][q], acc, 0, 0, 0);
  return acc;
}

// Householder QR of the w <= QW columns of A = W(p:, p:) (m2 rows, leading
// dimension ld), in dgeqrf's layout, and tau. One workgroup; thread t keeps
// rows t + 512 a of CW columns in registers, the panel's columns in QW / CW
// turns (a turn first applies the reflectors of the ones before it).
//
// Bound: the latency of a column's chain, and one barrier per column: the
// dot products of column j (rows below j) with every column held come from
// one reduction (a butterfly that halves the values a lane carries, then
// eight wave partials in LDS), and everything else follows from them and
// from row j: |x|^2 is one of them and v^T a_c = a_c(j) + s d_c for
// v = (1, s x). A lane forms one column's coefficient; the others read it
// from that lane. The column at hand is always register column 0 (a finished
// one is stored and the rest move down), so that the steps are loops and not
// QW copies of the code, which took five times as long, all of it
// instruction fetch.
template <int RPT, int CW>
struct QrPanel {
  double* A;
  double* tau;
  double* ts;                     // LDS: tau
  double (*red)[8][16];           // LDS [2]: wave partials
  double (*rowv)[16];             // LDS [2]: row j
  int ld, m2, w, t, lane, wave, buf;
  double x[RPT][CW];

  // sum over the workgroup of d[lane % NC], NC = 1 << LOG
  template <int LOG>
  __device__ __forceinline__ double reduce(double (&d)[1 << LOG]) {
    fold_halves<1 << LOG, 32>(d, lane);
    const double z = fold_sum<(32 >> LOG)>(d[0]);
    if ((lane & ((64 >> LOG) - 1)) == 0) red[buf][wave][lane >> (6 - LOG)] = z;
    __syncthreads();
    double g = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) g += red[buf][q][lane & ((1 << LOG) - 1)];
    return g;
  }

  // columns j0 .. j1 - 1, the 1 << LOG columns from j0 on in x
  template <int LOG>
  __device__ __forceinline__ void factor(int j0, int j1) {
    constexpr int NC = 1 << LOG;
    for (int j = j0; j < j1; ++j) {
      double g, rv, alpha, xn2, up = 1.0, down = 1.0;
      while (true) {
        double d[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) d[c] = 0.0;
#pragma unroll
        for (int a = 0; a < RPT; ++a) {
          const double xj = (a > 0 || t > j) ? x[a][0] : 0.0;
#pragma unroll
          for (int c = 0; c < NC; ++c) d[c] += xj * x[a][c];
        }
        if (t == j) {
#pragma unroll
          for (int c = 0; c < NC; ++c) rowv[buf][c] = x[0][c];
        }
        g = reduce<LOG>(d);
        rv = rowv[buf][lane & (NC - 1)];
        buf ^= 1;
        alpha = read_lane(rv, 0);
        xn2 = read_lane(g, 0);
        // the same in the whole workgroup
        if (!(xn2 < QR_TINY2) || !(fabs(alpha) * up < QR_TINY_PIVOT) || up > QR_UP) break;
#pragma unroll
        for (int a = 0; a < RPT; ++a)
          if (a > 0 || t > j) x[a][0] *= QR_UP;
        up *= QR_UP;
        down /= QR_UP;
      }
      double beta = alpha, tj = 0.0, scale = 0.0;
      if (!(xn2 < QR_TINY2) || (up > 1.0 && xn2 > 0.0)) {
        const double au = alpha * up, bu = -copysign(sqrt(au * au + xn2), au);
        beta = bu * down;
        tj = (bu - au) / bu;
        scale = 1.0 / (au - bu);
      }
      if (t == 0) {
        tau[j] = tj;
        ts[j] = tj;
      }
      const double f = tj * (rv + scale * g);
      double v[RPT];
#pragma unroll
      for (int a = 0; a < RPT; ++a) {
        const bool below = a > 0 || t > j;
        v[a] = below ? x[a][0] * scale : (t == j ? 1.0 : 0.0);
        const double s = below ? v[a] : (t == j ? beta : x[a][0]);
        if (t + 512 * a < m2) A[t + 512 * a + (size_t)j * ld] = s;
      }
#pragma unroll
      for (int c = 1; c < NC; ++c) {
        const double fc = read_lane(f, c);
#pragma unroll
        for (int a = 0; a < RPT; ++a) x[a][c - 1] = x[a][c] - fc * v[a];
      }
#pragma unroll
      for (int a = 0; a < RPT; ++a) x[a][NC - 1] = 0.0;
    }
  }

  // the reflector of an earlier column j, applied to the CW columns held
  template <int LOG>
  __device__ __forceinline__ void apply(int j) {
    double v[RPT], d[CW];
#pragma unroll
    for (int a = 0; a < RPT; ++a) v[a] = qr_v(A, ld, m2, w, t + 512 * a, j);
#pragma unroll
    for (int c = 0; c < CW; ++c) {
      d[c] = 0.0;
#pragma unroll
      for (int a = 0; a < RPT; ++a) d[c] += v[a] * x[a][c];
    }
    const double f = ts[j] * reduce<LOG>(d);
    buf ^= 1;
#pragma unroll
    for (int c = 0; c < CW; ++c) {
      const double fc = read_lane(f, c);
#pragma unroll
      for (int a = 0; a < RPT; ++a) x[a][c] -= fc * v[a];
    }
  }
};

// load(x, c0): columns c0 .. c0 + CW - 1 of the panel
template <int RPT, int CW, typename F>
__device__ __forceinline__ void qr_panel(double* A, int ld, int m2, int w, double* tau,
                                         F&& load) {
  __shared__ double red[2][8][16], rowv[2][16], ts[QW];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  QrPanel<RPT, CW> q;
  q.A = A;
  q.tau = tau;
  q.ts = ts;
  q.red = red;
  q.rowv = rowv;
  q.ld = ld;
  q.m2 = m2;
  q.w = w;
  q.t = t;
  q.lane = lane;
  q.wave = wave;
  q.buf = 0;
  for (int c0 = 0; c0 < w; c0 += CW) {
    load(q.x, c0);
    constexpr int LOG = CW == 16 ? 4 : CW == 8 ? 3 : 2;
    for (int j = 0; j < c0; ++j) q.template apply<LOG>(j);
    // the columns in hand halve as they are finished
    int j = c0;
    if constexpr (LOG >= 4) {
      q.template factor<4>(j, min(w, j + 8));
      j += 8;
    }
    if constexpr (LOG >= 3) {
      if (j < w) q.template factor<3>(j, min(w, j + 4));
      j += 4;
    }
    if (j < w) q.template factor<2>(j, min(w, j + 4));
    __syncthreads();   // the next turn reads what was stored
  }
}

template <int RPT, int CW>
__global__ __launch_bounds__(512) void qr_panel_kernel(double* __restrict__ A, int ld, int m2,
                                                       int w, double* __restrict__ tau) {
  qr_panel<RPT, CW>(A, ld, m2, w, tau, [&](double (&x)[RPT][CW], int c0) {
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int a = 0; a < RPT; ++a)
        x[a][c] = qr_c(A, ld, m2, w, (int)threadIdx.x + 512 * a, c0 + c);
  });
}

// C <- H^T C, H = H_0 ... H_{w-1} = I - V T V^T of the panel in A (m2 rows), in
// two launches over 256 rows x 16 columns per workgroup: partials of Y = V^T C,
// and of G = V^T V as one more column block; then X = T^T Y and C -= V X. T is
// not formed: T^-1 = diag(1 / tau) + the upper triangle of G, so X comes from
// substitution, x_i = tau_i (y_i - sum_{k<i} G(k, i) x_k). A memory
// round trip bounds either launch (the matrix is in the Infinity Cache, not
// in the writer's L2), so a wave's loads all go out together and the grid
// spans rows as well as columns: one workgroup per 16 columns, walking the
// rows, took 42 us a panel against 9 + 14 (2000 x 1000).
constexpr int QR_ROWS = 256;

__global__ __launch_bounds__(256) void qr_y_kernel(const double* __restrict__ A, int ld, int m2,
                                                   int w, const double* __restrict__ C, int ldc,
                                                   int nc, double* __restrict__ Yp) {
  __shared__ double ys[4][QW * 16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int b = (int)blockIdx.y * QR_ROWS + 64 * wave;
  d4v_t acc = {0.0, 0.0, 0.0, 0.0};
  if (blockIdx.x + 1 < gridDim.x) {
    const int cols = min(16, nc - (int)blockIdx.x * 16);
    C += (size_t)blockIdx.x * 16 * ldc;
    acc = qr_vt_c(A, ld, m2, w, b, lr, lg, acc,
                  [&](int l, int c) { return qr_c(C, ldc, m2, cols, l, c); });
  } else {
    acc = qr_vt_c(A, ld, m2, w, b, lr, lg, acc,
                  [&](int l, int c) { return qr_v(A, ld, m2, w, l, c); });
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) ys[wave][(4 * r + lg) + QW * lr] = acc[r];
  __syncthreads();
  Yp[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + t] =
      (ys[0][t] + ys[1][t]) + (ys[2][t] + ys[3][t]);
}

// -X(i, c) of columns 16 cb .. into xs (i + QW c), from the ns partials of Y
// and G; LDS ys, gs and ts, blocks of at least 256 threads
__device__ __forceinline__ void qr_coefficients(const double* __restrict__ Yp, int cb, int nb,
                                                int ns, int w, const double* __restrict__ tau,
                                                double* ys, double* gs, double* ts, double* xs) {
  const int t = threadIdx.x;
  if (t < QW) ts[t] = t < w ? tau[t] : 0.0;
  if (t < 256) {
    double y = 0.0, g = 0.0;
    for (int q0 = 0; q0 < ns; q0 += 8) {
      double yq[8], gq[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const size_t s = min(q0 + q, ns - 1);
        yq[q] = Yp[(s * (nb + 1) + cb) * 256 + t];
        gq[q] = Yp[(s * (nb + 1) + nb) * 256 + t];
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (q0 + q < ns) {
          y += yq[q];
          g += gq[q];
        }
    }
    ys[t] = y;
    gs[t] = g;
  }
  __syncthreads();
  if (t < 16) {
    double x[QW];   // y, less the terms of the x found so far
#pragma unroll
    for (int i = 0; i < QW; ++i) x[i] = ys[i + QW * t];
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      x[i] *= ts[i];
#pragma unroll
      for (int k = i + 1; k < QW; ++k) x[k] -= gs[i + QW * k] * x[i];
    }
#pragma unroll
    for (int i = 0; i < QW; ++i) xs[i + QW * t] = -x[i];
  }
  __syncthreads();
}

// rows b0 .. b0 + 63 of A's panel and of a 16-column block of C for one wave:
// loads and stores run along the rows (the product is issued transposed)
struct QrRows {
  double vb[4][4];
  d4v_t z[4];   // C(l, 4 r + lg)
  __device__ __forceinline__ void load(const double* __restrict__ A, int ld, int m2, int w,
                                       const double* C, int ldc, int cols, int b0, int lr, int lg) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        vb[u][q] = qr_v(A, ld, m2, w, b0 + 16 * u + lr, 4 * q + lg);
        z[u][q] = qr_c(C, ldc, m2, cols, b0 + 16 * u + lr, 4 * q + lg);
      }
  }
  __device__ __forceinline__ void update(const double* xs, double* C, int ldc, int m2, int cols,
                                         int b0, int lr, int lg) {
    double xa[4];   // -X(4 q + lg, lr), the left operand X^T(column, k)
#pragma unroll
    for (int q = 0; q < 4; ++q) xa[q] = xs[(4 * q + lg) + QW * lr];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int l = b0 + 16 * u + lr;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        z[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[q], vb[u][q], z[u], 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (l < m2 && 4 * r + lg < cols) C[l + (size_t)(4 * r + lg) * ldc] = z[u][r];
    }
  }
};

__global__ __launch_bounds__(256) void qr_update_kernel(const double* __restrict__ A, int ld,
                                                        int m2, int w,
                                                        const double* __restrict__ tau,
                                                        double* C, int ldc, int nc,
                                                        const double* __restrict__ Yp) {
  __shared__ double ys[QW * 16], gs[QW * QW], xs[QW * 16], ts[QW];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int cols = min(16, nc - (int)blockIdx.x * 16);
  const int b0 = (int)blockIdx.y * QR_ROWS + 64 * wave;
  C += (size_t)blockIdx.x * 16 * ldc;
  QrRows q;
  q.load(A, ld, m2, w, C, ldc, cols, b0, lr, lg);
  qr_coefficients(Yp, blockIdx.x, gridDim.x, gridDim.y, w, tau, ys, gs, ts, xs);
  q.update(xs, C, ldc, m2, cols, b0, lr, lg);
}

// The update, and the next panel (C's first block of columns, from row QW on)
// factored in the same launch: workgroup 0 updates that block in the registers
// it factors it in, while the others (512 rows x 16 columns each) update the
// rest. A panel takes longer than the update beside it (33 against 14 us),
// which is hidden: 34 us a panel, 2000 x 1000 3.92 -> 3.14 ms. The block's
// columns have to be the panel's: wn = min(QW, nc).
template <int RPT, int CW>
__global__ __launch_bounds__(512) void qr_step_kernel(const double* A, int ld, int m2,
                                                      const double* __restrict__ tau, double* C,
                                                      int nc, const double* __restrict__ Yp, int ns,
                                                      int wn, double* tau_next) {
  __shared__ double ys[QW * 16], gs[QW * QW], xs[QW * 16], ts[QW];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lr = lane & 15, lg = lane >> 4, nb = (nc + 15) / 16;
  if (blockIdx.x > 0) {
    const int nr = (m2 + 511) / 512;
    const bool top = blockIdx.x + 1 == gridDim.x;   // the panel's block: R's rows only
    const int cb = top ? 0 : 1 + ((int)blockIdx.x - 1) / nr;
    const int cols = min(16, nc - cb * 16);
    const int b0 = top ? 64 * wave : ((int)blockIdx.x - 1) % nr * 512 + 64 * wave;
    C += (size_t)cb * 16 * ld;
    QrRows q;
    q.load(A, ld, m2, QW, C, ld, cols, b0, lr, lg);
    qr_coefficients(Yp, cb, nb, ns, QW, tau, ys, gs, ts, xs);
    q.update(xs, C, ld, top ? min(QW, m2) : m2, cols, b0, lr, lg);
    return;
  }
  const int cols = min(16, nc);
  constexpr int VC = 8 / RPT;   // reflectors a turn
  qr_panel<RPT, CW>(C + QW, ld, m2 - QW, wn, tau_next, [&](double (&x)[RPT][CW], int c0) {
    // row QW + t + 512 a of the panel and of C; every load is clamped
    int l[RPT];
#pragma unroll
    for (int a = 0; a < RPT; ++a) l[a] = min(QW + t + 512 * a, m2 - 1);
#pragma unroll
    for (int c = 0; c < CW; ++c) {
      const double* cc = C + (size_t)min(c0 + c, cols - 1) * ld;
#pragma unroll
      for (int a = 0; a < RPT; ++a) x[a][c] = cc[l[a]];
    }
    if (c0 == 0) qr_coefficients(Yp, 0, nb, ns, QW, tau, ys, gs, ts, xs);
    double v[RPT][VC];
#pragma unroll
    for (int i = 0; i < VC; ++i)
#pragma unroll
      for (int a = 0; a < RPT; ++a) v[a][i] = A[l[a] + (size_t)i * ld];
    // VC reflectors a turn, the next turn's loads in flight
#pragma unroll 1
    for (int i0 = 0; i0 < QW; i0 += VC) {
      double vn[RPT][VC];
      const double* an = A + (size_t)min(i0 + VC, QW - VC) * ld;
#pragma unroll
      for (int i = 0; i < VC; ++i)
#pragma unroll
        for (int a = 0; a < RPT; ++a) vn[a][i] = an[l[a] + (size_t)i * ld];
#pragma unroll
      for (int c = 0; c < CW; ++c) {
#pragma unroll
        for (int i = 0; i < VC; ++i) {
          const double f = xs[i0 + i + QW * ((c0 + c) & 15)];
#pragma unroll
          for (int a = 0; a < RPT; ++a) x[a][c] += v[a][i] * f;
        }
        if (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // or every f is read up front
      }
#pragma unroll
      for (int a = 0; a < RPT; ++a)
#pragma unroll
        for (int i = 0; i < VC; ++i) v[a][i] = vn[a][i];
    }
#pragma unroll
    for (int a = 0; a < RPT; ++a)
#pragma unroll
      for (int c = 0; c < CW; ++c)
        if (QW + t + 512 * a >= m2 || c0 + c >= wn) x[a][c] = 0.0;
  });
}

__global__ void qr_init_q_kernel(int m, int r, double* __restrict__ Q) {
  int64_t tot = (int64_t)m * r;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x)
    Q[e] = ((e % m) == (e / m)) ? 1.0 : 0.0;
}

// columns j < r of W: the reflectors, v(j) = 1 stored and zeros above
__global__ void qr_unit_lower_kernel(int m, int r, double* __restrict__ W) {
  int64_t tot = (int64_t)m * r;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int i = (int)(e % m), j = (int)(e / m);
    if (i <= j) W[e] = i == j ? 1.0 : 0.0;
  }
}

__global__ void qr_extract_r_kernel(int m, int n, int r, const double* __restrict__ W,
                                    double* __restrict__ R) {
  int64_t tot = (int64_t)r * n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int i = (int)(e % r), c = (int)(e / r);
    R[e] = i <= c ? W[i + (size_t)c * m] : 0.0;
  }
}

// ------------------------------------------------------- one-sided Jacobi
__global__ __launch_bounds__(256) void jac_round_kernel(double* __restrict__ W, int m,
                                                        double* __restrict__ V, int nv, int ncols,
                                                        int N, int rnd, double tol,
                                                        double small2,
                                                        double* __restrict__ offs) {
  __shared__ double sh[3][4];
  int i = blockIdx.x;
  int p, q;
  if (i == 0) { p = rnd; q = N - 1; }
  else { p = (rnd + i) % (N - 1); q = (rnd - i + (N - 1)) % (N - 1); }
  if (p >= ncols || q >= ncols) return;
  double* a = W + (size_t)p * m;
  double* b = W + (size_t)q * m;
  double sa = 0.0, sb = 0.0, sg = 0.0;
  for (int r = threadIdx.x; r < m; r += blockDim.x) {
    double x = a[r], y = b[r];
    sa += x * x; sb += y * y; sg += x * y;
  }
  for (int o = 32; o > 0; o >>= 1) {
    sa += __shfl_down(sa, o, 64);
    sb += __shfl_down(sb, o, 64);
    sg += __shfl_down(sg, o, 64);
  }
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { sh[0][w] = sa; sh[1][w] = sb; sh[2][w] = sg; }
  __syncthreads();
  sa = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
  sb = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
  sg = sh[2][0] + sh[2][1] + sh[2][2] + sh[2][3];
  // a column at the rounding level of ||A||_F has no direction left to fix
  // (its cosines stay O(1) noise): such pairs count as converged
  double rel = (sa > small2 && sb > small2) ? fabs(sg) / sqrt(sa * sb) : 0.0;
  if (threadIdx.x == 0) offs[i] = fmax(offs[i], rel);
  if (rel <= tol) return;
  double zeta = (sb - sa) / (2.0 * sg);
  double t = copysign(1.0, zeta) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
  double c = 1.0 / sqrt(1.0 + t * t), s = c * t;
  for (int r = threadIdx.x; r < m; r += blockDim.x) {
    double x = a[r], y = b[r];
    a[r] = c * x - s * y;
    b[r] = s * x + c * y;
  }
  double* va = V + (size_t)p * nv;
  double* vb = V + (size_t)q * nv;
  for (int r = threadIdx.x; r < nv; r += blockDim.x) {
    double x = va[r], y = vb[r];
    va[r] = c * x - s * y;
    vb[r] = s * x + c * y;
  }
}

// ------------------------------------- orthogonalising nearly orthogonal columns
// G = W^T W of columns that a preceding eigenbasis left nearly orthogonal.
// A pair (i, j), i < j, is converged as in jac_round_kernel: its cosine is
// within tol, or a column is at the rounding level of ||A||. Any other is
// turned by the angle theta = atan(2 g_ij / (g_jj - g_ii)) / 2 that
// annihilates it; all small angles are applied at once as a matrix product
// (columns W X, X = I + K + K^2/2, K antisymmetric), which squares the
// cosines like a Jacobi sweep. Pairs at a larger angle (near-equal columns,
// or columns whose directions the eigenbasis did not resolve) are left for
// a new eigenbasis of the columns from the first of them on.
constexpr double ORTHO_ANGLE = 0.02;   // largest angle turned by K

__device__ __forceinline__ bool ortho_pair(const double* __restrict__ G, int n, int i, int j,
                                           double tol, double small2, double* rel,
                                           double* theta) {
  const double gi = G[(size_t)i * n + i], gj = G[(size_t)j * n + j];
  const double g = G[(size_t)j * n + i];
  *rel = (gi > small2 && gj > small2) ? fabs(g) / sqrt(gi * gj) : 0.0;
  if (*rel <= tol) return false;
  const double dd = gj - gi;
  // |theta| <= pi / 4: the pair's order is kept when the two are equal
  *theta = dd == 0.0 ? copysign(0.78539816339744831, g) : 0.5 * atan(2.0 * g / dd);
  return true;
}

// stat[0] = largest cosine (bits of a non-negative double), stat[1] = first
// index of a pair at a large angle (initialised to 0 and n); exact, so the
// order of the atomics does not matter
__global__ __launch_bounds__(256) void ortho_stat_kernel(const double* __restrict__ G, int n,
                                                         double tol, double small2,
                                                         unsigned long long* stat) {
  const int64_t tot = (int64_t)n * n;
  double mx = 0.0;
  int first = n;
  for (int64_t e = blockIdx.x * 256LL + threadIdx.x; e < tot; e += (int64_t)gridDim.x * 256) {
    const int i = (int)(e % n), j = (int)(e / n);
    if (i >= j) continue;
    double rel, th;
    if (ortho_pair(G, n, i, j, tol, small2, &rel, &th) && fabs(th) > ORTHO_ANGLE)
      first = min(first, i);
    mx = fmax(mx, rel);
  }
  for (int o = 32; o > 0; o >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, o, 64));
    first = min(first, __shfl_xor(first, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    atomicMax(stat, (unsigned long long)__double_as_longlong(mx));
    if (first < n) atomicMin(stat + 1, (unsigned long long)first);
  }
}

__global__ void ortho_init_kernel(int n, unsigned long long* stat) {
  stat[0] = 0;
  stat[1] = (unsigned long long)n;
}

// K over the pairs with i < first (stat[1]) and per-block partials of its
// squared norm
__global__ __launch_bounds__(256) void ortho_k_kernel(const double* __restrict__ G, int n,
                                                      double tol, double small2,
                                                      const unsigned long long* stat,
                                                      double* __restrict__ K,
                                                      double* __restrict__ part) {
  __shared__ double sh4[4];
  const int first = (int)stat[1];
  const int64_t tot = (int64_t)n * n;
  double s = 0.0;
  for (int64_t e = blockIdx.x * 256LL + threadIdx.x; e < tot; e += (int64_t)gridDim.x * 256) {
    const int r = (int)(e % n), c = (int)(e / n);
    const int i = min(r, c), j = max(r, c);
    double rel, th, v = 0.0;
    if (i != j && i < first && ortho_pair(G, n, i, j, tol, small2, &rel, &th) &&
        fabs(th) <= ORTHO_ANGLE)
      v = r < c ? th : -th;
    K[e] = v;
    s += v * v;
  }
  s = block_sum256(s, sh4);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// X = X + a I + b Y
__global__ void add_diag_kernel(int n, double a, double b, const double* __restrict__ Y,
                                double* __restrict__ X) {
  const int64_t tot = (int64_t)n * n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    double v = X[e] + (Y ? b * Y[e] : 0.0);
    if (e % n == e / n) v += a;
    X[e] = v;
  }
}

__global__ __launch_bounds__(256) void col_norm_kernel(const double* __restrict__ W, int m, int ncols,
                                                       double* __restrict__ out) {
  int lane = threadIdx.x & 63;
  int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= ncols) return;
  const double* col = W + (size_t)c * m;
  double s = 0.0;
  for (int r = lane; r < m; r += 64) s += col[r] * col[r];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) out[c] = sqrt(s);
}

__global__ void square_kernel(int n, const double* __restrict__ x, double* __restrict__ y) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i] * x[i];
}

// Uo[:, i] = W[:, perm[i]] / s_i (zero column if s_i == 0), Vo[:, i] = V[:, perm[i]]
__global__ void svd_gather_kernel(int m, int nv, int k, const double* __restrict__ W,
                                  const double* __restrict__ V, const int* __restrict__ perm,
                                  const double* __restrict__ s, double* __restrict__ Uo,
                                  double* __restrict__ Vo, int ldu, int ldv) {
  int64_t tot = (int64_t)(m > nv ? m : nv) * k;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t rows = m > nv ? m : nv;
    int r = (int)(e % rows), i = (int)(e / rows);
    int c = perm[i];
    if (r < m) Uo[r + (size_t)i * ldu] = s[i] > 0.0 ? W[r + (size_t)c * m] / s[i] : 0.0;
    if (r < nv) Vo[r + (size_t)i * ldv] = V[r + (size_t)c * nv];
  }
}

__global__ void transpose_kernel(int m, int n, const double* __restrict__ A, double* __restrict__ B) {
  int64_t tot = (int64_t)m * n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * blockDim.x) {
    int i = (int)(e % m), j = (int)(e / m);
    B[j + (size_t)i * n] = A[e];
  }
}

}  // namespace

// doubles of the partials of V^T C (nc columns) and V^T V
static size_t qr_yp_doubles(int m, int nc) {
  return (size_t)((m + QR_ROWS - 1) / QR_ROWS) * ((nc + 15) / 16 + 1) * 256;
}

// W (m x n, m <= QR_MAX_ROWS) <- its QR in dgeqrf's layout; Yp holds
// qr_yp_doubles(m, n)
static int qr_blocked(itg_ctx* ctx, int m, int n, double* W, double* tau, double* Yp) {
  const int r = std::min(m, n);
  hipStream_t st = ctx->stream;
  // rows a thread x columns a turn: at most 64 doubles of the panel
  auto panel = [&](double* A, int rows, int w, double* tp) {
    if (rows <= 1024) qr_panel_kernel<2, 16><<<1, 512, 0, st>>>(A, m, rows, w, tp);
    else if (rows <= 2048) qr_panel_kernel<4, 16><<<1, 512, 0, st>>>(A, m, rows, w, tp);
    else if (rows <= 4096) qr_panel_kernel<8, 8><<<1, 512, 0, st>>>(A, m, rows, w, tp);
    else qr_panel_kernel<16, 4><<<1, 512, 0, st>>>(A, m, rows, w, tp);
  };
  panel(W, m, std::min(QW, r), tau);
  ITG_LAUNCH_CHECK(ctx);
  for (int p = 0; p < r; p += QW) {
    const int w = std::min(QW, r - p), m2 = m - p, nt = n - p - w;
    if (nt <= 0) break;
    double* A = W + (size_t)p * m + p;
    double* C = A + (size_t)w * m;
    const int nb = (nt + 15) / 16, ns = (m2 + QR_ROWS - 1) / QR_ROWS;
    qr_y_kernel<<<dim3(nb + 1, ns), 256, 0, st>>>(A, m, m2, w, C, m, nt, Yp);
    const int pn = p + QW, rows = m - pn, wn = std::min(QW, r - pn);
    auto step = [&](auto kernel) {
      kernel<<<2 + (nb - 1) * ((m2 + 511) / 512), 512, 0, st>>>(A, m, m2, tau + p, C, nt, Yp, ns, wn,
                                                                tau + pn);
    };
    // past 4096 rows the panel's registers leave no room for the update; and a
    // last panel narrower than its block of columns (a wide matrix) leaves
    // columns of the block that the panel's workgroup does not hold
    if (wn < std::min(QW, nt) || rows > 4096) {
      qr_update_kernel<<<dim3(nb, ns), 256, 0, st>>>(A, m, m2, w, tau + p, C, m, nt, Yp);
      if (wn > 0) panel(C + QW, rows, wn, tau + pn);
    } else if (rows <= 1024) {
      step(qr_step_kernel<2, 16>);
    } else if (rows <= 2048) {
      step(qr_step_kernel<4, 16>);
    } else {
      step(qr_step_kernel<8, 8>);
    }
    ITG_LAUNCH_CHECK(ctx);
  }
  return ITG_OK;
}

extern "C" int itg_qr(itg_ctx* ctx, int dtype, int64_t m64, int64_t n64, const void* Ain, void* Qo,
                      void* Ro) {
  ITG_CHECK_CTX(ctx);
  if (dtype != ITG_C64) ITG_CHECK_DTYPE(ctx, dtype);
  if (m64 < 0 || n64 < 0) return itg_fail(ctx, ITG_EDIM, "qr: negative dimension");
  if (m64 * n64 > ((int64_t)1 << 31)) return itg_fail(ctx, ITG_EUNSUPPORTED, "qr: matrix too large");
  if (m64 == 0 || n64 == 0) return ITG_OK;
  if (dtype == ITG_C64) return itg_c64_qr(ctx, m64, n64, Ain, Qo, Ro);
  int m = (int)m64, n = (int)n64, r = std::min(m, n);
  const size_t nx = std::max((size_t)NB * n, (size_t)BT_GROUP * r);
  size_t bytes = ((size_t)m * n + (size_t)m * r + (size_t)r * n + (size_t)m * NB + 2 * nx +
                  (size_t)BT_GROUP * BT_GROUP + NB * NB + (size_t)r +
                  (m <= QR_MAX_ROWS ? qr_yp_doubles(m, n) : 0) + 64) * sizeof(double) + 16 * 256;
  void* ws;
  int rc = eig_workspace(ctx, bytes, &ws);
  if (rc) return rc;
  Carver cv{(char*)ws};
  double* W = cv.take<double>((size_t)m * n);
  double* Q = cv.take<double>((size_t)m * r);
  double* R = cv.take<double>((size_t)r * n);
  double* Vb = cv.take<double>((size_t)m * NB);
  double* X = cv.take<double>(nx);
  double* X2 = cv.take<double>(nx);
  double* Gm = cv.take<double>((size_t)BT_GROUP * BT_GROUP);
  double* Tm = cv.take<double>(NB * NB);
  double* tau = cv.take<double>(r);
  rc = itg_convert(ctx, (int64_t)m * n, dtype, Ain, ITG_F64, W);
  if (rc) return rc;
  if (m <= QR_MAX_ROWS) {
    rc = qr_blocked(ctx, m, n, W, tau, cv.take<double>(qr_yp_doubles(m, n)));
    if (rc) return rc;
  }
  // taller matrices: blocked Householder QR (dgeqrf): each panel of NB columns is factored
  // column by column within itself, then the trailing columns take the
  // panel's block reflector, W2 -= V T^T (V^T W2), as GEMMs
  for (int p = 0; p < r && m > QR_MAX_ROWS; p += NB) {
    const int nbp = std::min(NB, r - p), pe = p + nbp;
    for (int j = p; j < pe; ++j) {
      qr_reflect_kernel<<<1, 1024, 0, ctx->stream>>>(W, m, j, tau);
      if (j + 1 < pe)
        qr_apply_kernel<<<pe - j - 1, 256, 0, ctx->stream>>>(W, m, pe, j, tau);
      ITG_LAUNCH_CHECK(ctx);
    }
    const int nt = n - pe, m2 = m - p;
    if (nt <= 0) continue;
    bt_build_v_kernel<<<itg_blocks((int64_t)m * nbp, 256, 4096), 256, 0, ctx->stream>>>(W, m, p, nbp,
                                                                                         0, Vb);
    ITG_LAUNCH_CHECK(ctx);
    const double* V1 = Vb + p;
    double* W2 = W + (size_t)pe * m + p;
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', nbp, nbp, m2, 1.0, V1, m, V1,
                           m, 0.0, Gm, nbp);
    if (rc) return rc;
    bt_larft_kernel<<<1, 64, 0, ctx->stream>>>(nbp, Gm, tau + p, Tm);
    ITG_LAUNCH_CHECK(ctx);
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', nbp, nt, m2, 1.0, V1, m, W2,
                           m, 0.0, X, nbp);
    if (rc) return rc;
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', nbp, nt, nbp, 1.0, Tm, nbp, X,
                           nbp, 0.0, X2, nbp);
    if (rc) return rc;
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', m2, nt, nbp, -1.0, V1, m, X2,
                           nbp, 1.0, W2, m);
    if (rc) return rc;
  }
  qr_extract_r_kernel<<<itg_blocks((int64_t)r * n, 256, 8192), 256, 0, ctx->stream>>>(m, n, r, W, R);
  qr_unit_lower_kernel<<<itg_blocks((int64_t)m * r, 256, 8192), 256, 0, ctx->stream>>>(m, r, W);
  qr_init_q_kernel<<<itg_blocks((int64_t)m * r, 256, 8192), 256, 0, ctx->stream>>>(m, r, Q);
  ITG_LAUNCH_CHECK(ctx);
  rc = back_transform_groups(ctx, m, r, 0, r, W, tau, Q, true, X, X2, Gm);
  if (rc) return rc;
  rc = itg_convert(ctx, (int64_t)m * r, ITG_F64, Q, dtype, Qo);
  if (rc) return rc;
  return itg_convert(ctx, (int64_t)r * n, ITG_F64, R, dtype, Ro);
}

// Buffers of ortho_columns: W and V with a second buffer each (swapped as
// they are rotated), and three n x n matrices.
struct OrthoBufs {
  double *W, *W2, *V, *V2, *G, *K, *X, *wG;
  double* part;               // 1024 partials
  unsigned long long* stat;   // 2
};

// Makes the columns of W (rows x n, already W = A V with V an eigenbasis of
// A^T A, columns by descending norm) orthogonal to tol by rotations applied
// to W and V alike: matrix products while every angle is small, a new
// eigenbasis of the trailing columns where one is not. *done is false if
// some pair has to be left to the Jacobi sweeps.
//
// Against the sweeps alone: a sweep is n - 1 launches of n / 2 column pairs,
// ~10 us each whatever they do (2 sweeps, 40 ms, at 2048 x 2048, and one
// more to see that nothing is left); a pass here is one Gram product and, if
// it turns anything, four to six more of the same size (0.25 to 0.35 ms each).
int ortho_columns(itg_ctx* ctx, int rows, int n, double tol, double small2, OrthoBufs& b,
                  bool* done) {
  constexpr int PARTS = 1024;
  *done = false;
  int64_t fresh = 0;   // columns given a new eigenbasis so far
  const unsigned gb = (unsigned)itg_blocks((int64_t)n * n, 256, PARTS);
  for (int pass = 0; pass < 14; ++pass) {
    int rc = itg_gemm(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', n, n, rows, 1.0, b.W, rows, b.W,
                      rows, 0.0, b.G, n);
    if (rc) return rc;
    ortho_init_kernel<<<1, 1, 0, ctx->stream>>>(n, b.stat);
    ortho_stat_kernel<<<gb, 256, 0, ctx->stream>>>(b.G, n, tol, small2, b.stat);
    ortho_k_kernel<<<gb, 256, 0, ctx->stream>>>(b.G, n, tol, small2, b.stat, b.K, b.part);
    ITG_LAUNCH_CHECK(ctx);
    unsigned long long st[2];
    std::vector<double> part(gb);
    ITG_HIP(ctx, hipMemcpyAsync(st, b.stat, sizeof st, hipMemcpyDeviceToHost, ctx->stream));
    ITG_HIP(ctx, hipMemcpyAsync(part.data(), b.part, gb * sizeof(double), hipMemcpyDeviceToHost,
                                ctx->stream));
    ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    double mx, kf = 0.0;
    memcpy(&mx, &st[0], sizeof mx);
    for (double x : part) kf += x;
    kf = std::sqrt(kf);
    if (mx <= tol) {
      *done = true;
      return ITG_OK;
    }
    const int first = (int)st[1];
    // X^T X - I = K^4 / 4 for X = I + K + K^2 / 2; each polishing step
    // X (3 I - X^T X) / 2 squares it
    if (!(kf <= 0.3)) return ITG_OK;
    // the trailing columns' scale: the eigensolver's deflation is absolute
    // below unit norm
    double gf = 1.0;
    if (first < n) {
      ITG_HIP(ctx, hipMemcpyAsync(&gf, b.G + (size_t)first * n + first, sizeof(double),
                                  hipMemcpyDeviceToHost, ctx->stream));
      ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    if (kf > 0.0) {
      rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', n, n, n, 0.5, b.K, n, b.K, n,
                             0.0, b.X, n);
      if (rc) return rc;
      add_diag_kernel<<<gb, 256, 0, ctx->stream>>>(n, 1.0, 1.0, b.K, b.X);
      for (int q = kf <= 1e-4 ? 0 : kf <= 1e-2 ? 1 : 2; q > 0; --q) {
        rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', n, n, n, -0.5, b.X, n, b.X,
                               n, 0.0, b.K, n);
        if (rc) return rc;
        add_diag_kernel<<<gb, 256, 0, ctx->stream>>>(n, 1.5, 0.0, nullptr, b.K);
        rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', n, n, n, 1.0, b.X, n, b.K,
                               n, 0.0, b.G, n);
        if (rc) return rc;
        std::swap(b.X, b.G);
      }
      rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', rows, n, n, 1.0, b.W, rows,
                             b.X, n, 0.0, b.W2, rows);
      if (rc) return rc;
      rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', n, n, n, 1.0, b.V, n, b.X, n,
                             0.0, b.V2, n);
      if (rc) return rc;
      std::swap(b.W, b.W2);
      std::swap(b.V, b.V2);
    }
    if (first < n) {
      // a spectrum over the whole range of a double takes about 1.5 n (each
      // new basis resolves seven digits and disturbs the next ones a little)
      const int t = n - first;
      fresh += t;
      if (fresh > 6 * (int64_t)n) return ITG_OK;
      const size_t wo = (size_t)first * rows, vo = (size_t)first * n;
      rc = itg_gemm(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', t, t, rows,
                    std::ldexp(1.0, std::min(1023, -std::ilogb(gf))), b.W + wo, rows, b.W + wo, rows,
                    0.0, b.G, t);
      if (rc) return rc;
      int64_t kg = 0;
      double teg = 0.0, dcg = 0.0;
      rc = itg_eigh_trunc(ctx, ITG_F64, t, b.G, b.wG, b.X, 0, -1.0, 0, 1, &kg, &teg, &dcg);
      if (rc) return rc;
      rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', rows, t, t, 1.0, b.W + wo,
                             rows, b.X, t, 0.0, b.W2 + wo, rows);
      if (rc) return rc;
      rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', n, t, t, 1.0, b.V + vo, n,
                             b.X, t, 0.0, b.V2 + vo, n);
      if (rc) return rc;
      ITG_HIP(ctx, hipMemcpyAsync(b.W2, b.W, wo * sizeof(double), hipMemcpyDeviceToDevice,
                                  ctx->stream));
      ITG_HIP(ctx, hipMemcpyAsync(b.V2, b.V, vo * sizeof(double), hipMemcpyDeviceToDevice,
                                  ctx->stream));
      std::swap(b.W, b.W2);
      std::swap(b.V, b.V2);
    }
  }
  return ITG_OK;
}

// smallest column count at which the Jacobi SVD is preconditioned by the
// Gram matrix's eigenvectors
constexpr int SVD_PRECOND_MIN = 64;

extern "C" int itg_svd_trunc(itg_ctx* ctx, int dtype, int64_t m64, int64_t n64, void* Ain, void* Uo,
                             double* So, void* Vo, int64_t maxdim, int64_t mindim, double cutoff,
                             int abs_cut, int rel_cut, int64_t* kout, double* truncerr,
                             double* docut) {
  ITG_CHECK_CTX(ctx);
  if (dtype != ITG_C64) ITG_CHECK_DTYPE(ctx, dtype);
  if (m64 < 0 || n64 < 0) return itg_fail(ctx, ITG_EDIM, "svd: negative dimension");
  if (!kout) return itg_fail(ctx, ITG_EARG, "svd: null k");
  if (m64 == 0 || n64 == 0) {
    *kout = 0;
    if (truncerr) *truncerr = 0.0;
    if (docut) *docut = 0.0;
    return ITG_OK;
  }
  if (dtype == ITG_C64)
    return itg_c64_svd_trunc(ctx, m64, n64, Ain, Uo, So, Vo, maxdim, mindim, cutoff, abs_cut,
                             rel_cut, kout, truncerr, docut);
  if (std::min(m64, n64) > 8192 || m64 * n64 > ((int64_t)1 << 31))
    return itg_fail(ctx, ITG_EUNSUPPORTED, "svd: matrix too large");
  int rc = set_lds_limit(ctx);
  if (rc) return rc;
  int m = (int)m64, n = (int)n64;
  bool tr = m < n;                 // work on A^T so that rows >= cols
  int rows = tr ? n : m, cols = tr ? m : n;
  int N = cols + (cols & 1);
  // preconditioning (below) runs the eigensolver, which owns eig_ws: the
  // SVD's buffers live in their own grow-only workspace
  const bool precond = cols >= SVD_PRECOND_MIN;
  size_t bytes = ((size_t)rows * cols * 2 + (size_t)cols * cols + (size_t)rows * cols +
                  (size_t)cols * cols + 8 * (size_t)N + 64) * sizeof(double) + 16 * 256 +
                 (precond ? ((size_t)rows * cols + 4 * (size_t)cols * cols + cols + 1024 + 2) * 8 +
                                8 * 256
                          : 0);
  if (bytes > ctx->svd_ws_bytes) {
    if (ctx->svd_ws) {
      ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
      ITG_HIP(ctx, hipFree(ctx->svd_ws));
      ctx->svd_ws = nullptr;
      ctx->svd_ws_bytes = 0;
    }
    if (hipMalloc(&ctx->svd_ws, bytes) != hipSuccess) {
      hipGetLastError();
      return itg_fail(ctx, ITG_EOOM, "svd workspace of %zu bytes failed", bytes);
    }
    ctx->svd_ws_bytes = bytes;
  }
  void* ws = ctx->svd_ws;
  Carver cv{(char*)ws};
  double* A64 = cv.take<double>((size_t)m * n);
  double* W = cv.take<double>((size_t)rows * cols);
  double* V = cv.take<double>((size_t)cols * cols);
  double* Ub = cv.take<double>((size_t)rows * cols);
  double* Vbo = cv.take<double>((size_t)cols * cols);
  double* offs = cv.take<double>(N);
  double* sig = cv.take<double>(N);
  double* sig_sorted = cv.take<double>(N);
  double* P = cv.take<double>(N);
  int* perm = cv.take<int>(N);
  double* out3 = cv.take<double>(4);
  rc = itg_convert(ctx, (int64_t)m * n, dtype, Ain, ITG_F64, A64);
  if (rc) return rc;
  if (tr) transpose_kernel<<<itg_blocks((int64_t)m * n, 256, 8192), 256, 0, ctx->stream>>>(m, n, A64, W);
  else ITG_HIP(ctx, hipMemcpyAsync(W, A64, (size_t)m * n * 8, hipMemcpyDeviceToDevice, ctx->stream));
  OrthoBufs ob = {};
  if (precond) {
    // Jacobi preconditioned by the Gram matrix's eigenvectors: W <- W V0
    // with W^T W = V0 diag(w) V0^T, V <- V0. The columns of W V0 are
    // orthogonal up to eps ||A||^2 / (s_i s_j); ortho_columns turns what is
    // left by matrix products, and the one-sided sweeps below take over
    // where it cannot finish
    double* G = cv.take<double>((size_t)cols * cols);
    double* W2 = cv.take<double>((size_t)rows * cols);
    double* wG = cv.take<double>(cols);
    ob = {W2, W, V, cv.take<double>((size_t)cols * cols), G, cv.take<double>((size_t)cols * cols),
          cv.take<double>((size_t)cols * cols), wG, cv.take<double>(1024),
          cv.take<unsigned long long>(2)};
    if (cv.off > bytes) return itg_fail(ctx, ITG_EOOM, "svd: workspace layout overflow");
    // (one operand buffer: the exactly symmetric product)
    rc = itg_gemm(ctx, ITG_F64, ITG_MODE_NATIVE, 'T', 'N', cols, cols, rows, 1.0, W, rows, W, rows,
                  0.0, G, cols);
    if (rc) return rc;
    int64_t kg = 0;
    double teg = 0.0, dcg = 0.0;
    rc = itg_eigh_trunc(ctx, ITG_F64, cols, G, wG, V, 0, -1.0, 0, 1, &kg, &teg, &dcg);
    if (rc) return rc;
    rc = itg_gemm_internal(ctx, ITG_F64, ITG_MODE_NATIVE, 'N', 'N', rows, cols, cols, 1.0, W, rows,
                           V, cols, 0.0, W2, rows);
    if (rc) return rc;
  } else {
    qr_init_q_kernel<<<itg_blocks((int64_t)cols * cols, 256, 8192), 256, 0, ctx->stream>>>(cols, cols, V);
    ITG_LAUNCH_CHECK(ctx);
  }
  double tol = 4.0 * ITG_DC_EPS * std::sqrt((double)rows);
  double fro = 0.0;
  rc = itg_nrm2(ctx, ITG_F64, (int64_t)m * n, A64, &fro);
  if (rc) return rc;
  double small2 = (ITG_DC_EPS * fro) * (ITG_DC_EPS * fro);
  std::vector<double> hoffs(N / 2);
  bool conv = cols < 2;
  if (precond) {
    rc = ortho_columns(ctx, rows, cols, tol, small2, ob, &conv);
    if (rc) return rc;
    W = ob.W;
    V = ob.V;
  }
  for (int sweep = 0; sweep < 60 && !conv; ++sweep) {
    ITG_HIP(ctx, hipMemsetAsync(offs, 0, (N / 2) * sizeof(double), ctx->stream));
    for (int rnd = 0; rnd < N - 1; ++rnd) {
      jac_round_kernel<<<N / 2, 256, 0, ctx->stream>>>(W, rows, V, cols, cols, N, rnd, tol, small2,
                                                       offs);
    }
    ITG_LAUNCH_CHECK(ctx);
    ITG_HIP(ctx, hipMemcpyAsync(hoffs.data(), offs, (N / 2) * sizeof(double),
                                hipMemcpyDeviceToHost, ctx->stream));
    ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    double mx = 0.0;
    for (double x : hoffs) mx = std::max(mx, x);
    conv = mx <= tol;
  }
  if (!conv) return itg_fail(ctx, ITG_ECONV, "svd: Jacobi sweeps did not converge");
  col_norm_kernel<<<(cols + 3) / 4, 256, 0, ctx->stream>>>(W, rows, cols, sig);
  int np2 = 1;
  while (np2 < cols) np2 <<= 1;
  dc_final_sort_kernel<<<1, 1024, (size_t)np2 * 12, ctx->stream>>>(cols, sig, perm, sig_sorted);
  square_kernel<<<(cols + 255) / 256, 256, 0, ctx->stream>>>(cols, sig_sorted, P);
  ITG_LAUNCH_CHECK(ctx);
  rc = itg_truncate_device_async(ctx, P, cols, maxdim, mindim, cutoff, abs_cut, rel_cut,
                                 ITG_TRUNC_NDTENSORS, out3);
  if (rc) return rc;
  double h[3];
  ITG_HIP(ctx, hipMemcpyAsync(h, out3, 3 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  ITG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  int k = (int)h[0];
  svd_gather_kernel<<<itg_blocks((int64_t)std::max(rows, cols) * k, 256, 8192), 256, 0, ctx->stream>>>(
      rows, cols, k, W, V, perm, sig_sorted, Ub, Vbo, rows, cols);
  ITG_LAUNCH_CHECK(ctx);
  // A = Ub S Vbo^T (or its transpose)
  double* Ua = tr ? Vbo : Ub;   // m x k, ld m
  double* Va = tr ? Ub : Vbo;   // n x k, ld n
  rc = itg_convert(ctx, (int64_t)m * k, ITG_F64, Ua, dtype, Uo);
  if (rc) return rc;
  rc = itg_convert(ctx, (int64_t)n * k, ITG_F64, Va, dtype, Vo);
  if (rc) return rc;
  ITG_HIP(ctx, hipMemcpyAsync(So, sig_sorted, std::min(m, n) * sizeof(double), hipMemcpyDeviceToDevice,
                              ctx->stream));
  *kout = k;
  if (truncerr) *truncerr = h[1];
  if (docut) *docut = h[2];
  return ITG_OK;
}
