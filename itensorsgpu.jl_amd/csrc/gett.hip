// Tensor contraction C = alpha * A.B + beta * C on gfx950 MFMA, with every
// index permutation folded into the operand loads and the epilogue.
//
// The contraction is reduced to GEMM coordinates (m, n, k): m runs over the
// free modes of A, n over those of B, k over the contracted modes. The
// address of A(m,k) is offAm[m] + offAk[k] (likewise B, C); each offset is
// either affine (one merged mode: idx * stride) or read from a small table
// built on the host and cached per contraction signature, the analogue of
// the reference's ContractionPlans cache (src/ITensorsGPU.jl:55,
// src/tensor/cudense.jl:285-326). Tables replace the permutedims passes of
// the TTGT route (cudense.jl:170-236): tiles are gathered straight from the
// tensors into LDS, in whichever direction (m/n or k) is contiguous in HBM.
//
// 256-thread workgroups, 2x2 waves:
//   native : gett_native_kernel, 32 x 32 to 128 x 128 tiles,
//            v_mfma_f64_16x16x4_f64 (FP64 storage, FP64 accumulate) or
//            v_mfma_f32_16x16x4_f32 (FP32 storage, FP32 accumulate)
//   FP32 on FP64 storage, BF16x3 : gett_kernel, 128 x 128 tiles,
//            v_mfma_f32_16x16x4_f32; BF16x3 splits a = ah + al, b = bh + bl
//            (bf16, round-to-nearest-even) and sums ah*bh + ah*bl + al*bh on
//            v_mfma_f32_16x16x32_bf16, FP32 accumulate (Henry, Tang &
//            Heinecke, ARITH 2019)
// Workgroup ids are remapped so that each XCD (ids congruent mod 8) works on
// a contiguous group of tiles sharing A/B panels in its own L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <numeric>
#include <type_traits>

#include "itg_internal.h"

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

#include "gett.h"

__device__ __forceinline__ int64_t goff(const int64_t* t, int64_t s, int64_t i) {
  return s >= 0 ? i * s : t[i];
}

__device__ __forceinline__ uint16_t f2bf_rne(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

template <int MODE>
struct GettTraits {
  static constexpr bool BF = (MODE == ITG_MODE_BF16X3);
  static constexpr int BM = 128, BN = 128;
  static constexpr int BKT = BF ? 32 : 16;
  static constexpr int NPT = BM * BKT / 256;   // elements per thread per operand
};

// map workgroup id -> (tm, tn) with XCD-aware placement and grouped order
__device__ __forceinline__ void tile_coords(int64_t tilesM, int64_t tilesN, int64_t& tm,
                                            int64_t& tn) {
  int64_t nb = (int64_t)gridDim.x, bid = blockIdx.x;
  int64_t lid = bid;
  if (nb % 8 == 0) lid = (bid % 8) * (nb / 8) + bid / 8;
  const int64_t GM = 8;
  int64_t per_group = GM * tilesN;
  int64_t group = lid / per_group;
  int64_t first = group * GM;
  int64_t gsize = tilesM - first < GM ? tilesM - first : GM;
  int64_t in = lid % per_group;
  tm = first + in % gsize;
  tn = in / gsize;
}

// Band products (square C, tiles tm <= tn + 1 only): the live tiles alone are
// numbered, column by column, and each XCD takes an equal run of them. With
// the full grid's numbering the dead tiles left some XCDs idle, and half the
// work took as long as all of it (4096^3 FP64: 2240 us, 1240 now).
__host__ __device__ inline int64_t band_tiles(int64_t T) { return T * (T + 1) / 2 + T - 1; }
__device__ __forceinline__ bool band_coords(int64_t T, int64_t& tm, int64_t& tn) {
  const int64_t lid = (int64_t)(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  if (lid >= band_tiles(T)) return false;
  tn = (int64_t)((sqrt(9.0 + 8.0 * (double)lid) - 3.0) * 0.5);
  while (tn * (tn + 3) / 2 > lid) --tn;
  while ((tn + 1) * (tn + 4) / 2 <= lid) ++tn;
  tm = lid - tn * (tn + 3) / 2;
  return true;
}

// Epilogue of gett_kernel's 128 x 128 tile (2 x 2 waves of 4 x 4 blocks):
// lane holds D[4*lg + r][lr] of each 16x16 block
template <typename T>
__device__ __forceinline__ void gett_epilogue(const GettArgs& g, f4_t (&acc)[4][4], int64_t m0,
                                              int64_t n0, int wm, int wn, int lr, int lg) {
  constexpr int BM = 128, BN = 128, WH = 64, WT = 4;
  using CT = float;
  if (g.partial) {
    CT* P = (CT*)g.partial + (int64_t)blockIdx.z * g.M * g.N;
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int j = 0; j < WT; ++j) {
        int64_t n = n0 + wn * WH + j * 16 + lr;
        if (n >= g.N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int64_t m = m0 + wm * WH + i * 16 + 4 * lg + r;
          if (m < g.M) P[m * g.N + n] = acc[i][j][r];
        }
      }
    return;
  }
  T* C = (T*)g.C;
  if (g.sCm == 1 && g.sCn >= 0 && m0 + BM <= g.M && n0 + BN <= g.N) {
    // interior tile of a column-major C: one column pointer per j and
    // compile-time row offsets, no per-element bounds or offset arithmetic
    // (a short epilogue: this code runs once per tile, from a cold
    // instruction cache on small launches)
    T* cb = C + (n0 + wn * WH + lr) * g.sCn + m0 + wm * WH + 4 * lg;
    const double al = g.alpha, be = g.beta;
    if (be != 0.0) {
#pragma unroll
      for (int j = 0; j < WT; ++j) {
        T* cj = cb + (int64_t)(j * 16) * g.sCn;
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int mo = i * 16 + r;
            cj[mo] = (T)(al * (double)acc[i][j][r] + be * (double)cj[mo]);
          }
      }
    } else {
#pragma unroll
      for (int j = 0; j < WT; ++j) {
        T* cj = cb + (int64_t)(j * 16) * g.sCn;
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) cj[i * 16 + r] =
              (T)(al * (double)acc[i][j][r]);
      }
    }
    return;
  }
  if (g.sCn == 1 && g.sCm >= 0 && m0 + BM <= g.M && n0 + BN <= g.N) {
    // the same for a row-major C (itg_gemm's C^T): one row pointer per
    // (i, r), compile-time column offsets
    T* cb = C + (m0 + wm * WH + 4 * lg) * g.sCm + n0 + wn * WH + lr;
    const double al = g.alpha, be = g.beta;
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        T* ci = cb + (int64_t)(i * 16 + r) * g.sCm;
        if (be != 0.0) {
#pragma unroll
          for (int j = 0; j < WT; ++j)
            ci[j * 16] = (T)(al * (double)acc[i][j][r] + be * (double)ci[j * 16]);
        } else {
#pragma unroll
          for (int j = 0; j < WT; ++j) ci[j * 16] = (T)(al * (double)acc[i][j][r]);
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int j = 0; j < WT; ++j) {
      int64_t n = n0 + wn * WH + j * 16 + lr;
      if (n >= g.N) continue;
      int64_t on = goff(g.tCn, g.sCn, n);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int64_t m = m0 + wm * WH + i * 16 + 4 * lg + r;
        if (m >= g.M) continue;
        int64_t o = on + goff(g.tCm, g.sCm, m);
        double v = g.alpha * (double)acc[i][j][r];
        if (g.beta != 0.0) v += g.beta * (double)C[o];
        C[o] = (T)v;
      }
    }
}

template <typename T, int MODE, bool AK, bool BKF>
__global__ __launch_bounds__(256, 2) void gett_kernel(GettArgs g) {
  using TR = GettTraits<MODE>;
  using CT = float;
  constexpr int BM = TR::BM, BN = TR::BN, BKT = TR::BKT, NPT = TR::NPT;
  // four waves in 2 x 2, each a WH x WH sub-tile of WT x WT 16 x 16 blocks
  constexpr int WH = BM / 2, WT = BM / 32;
  constexpr bool BF = TR::BF;
  constexpr int PAD = BF ? 8 : 1;

  // LDS: FP64/FP32 k-major [k][m]; BF16 m-major [m][k] (8 consecutive k per lane)
  __shared__ __attribute__((aligned(16))) char smem[BF ? (4 * BM * (BKT + PAD) * 2)
                                                       : (2 * BKT * (BM + PAD) * sizeof(CT))];
  CT* As = (CT*)smem;
  CT* Bs = As + BKT * (BM + PAD);
  uint16_t* Ah = (uint16_t*)smem;
  uint16_t* Al = Ah + BM * (BKT + PAD);
  uint16_t* Bh = Al + BM * (BKT + PAD);
  uint16_t* Bl = Bh + BN * (BKT + PAD);

  const T* __restrict__ A = (const T*)g.A;
  const T* __restrict__ B = (const T*)g.B;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave & 1, wn = wave >> 1;

  int64_t tm, tn;
  tile_coords(g.tilesM, g.tilesN, tm, tn);
  if (g.band && tm > tn + 1) return;   // whole workgroup, before any barrier
  const int64_t m0 = tm * BM, n0 = tn * BN;
  const int64_t kbeg = (int64_t)blockIdx.z * g.kchunk;
  const int64_t kend = (kbeg + g.kchunk < g.K) ? kbeg + g.kchunk : g.K;

  // fixed per-thread coordinates for the loaders
  // A: AK ? (k = t % BKT, m = t / BKT + (256/BKT)*i) : (m = t % BM, k = t / BM + 2*i)
  constexpr int ASTEP = AK ? 256 / BKT : 256 / BM;
  constexpr int BSTEP = BKF ? 256 / BKT : 256 / BN;
  const int a_fix = AK ? (t % BKT) : (t % BM);
  const int a_var0 = AK ? (t / BKT) : (t / BM);
  const int b_fix = BKF ? (t % BKT) : (t % BN);
  const int b_var0 = BKF ? (t / BKT) : (t / BN);

  // offsets constant over the K loop
  int64_t a_offm[AK ? NPT : 1];
  int64_t b_offn[BKF ? NPT : 1];
  bool a_okm[AK ? NPT : 1];
  bool b_okn[BKF ? NPT : 1];
  if (AK) {
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      int64_t m = m0 + a_var0 + ASTEP * i;
      a_okm[i] = m < g.M;
      a_offm[i] = a_okm[i] ? goff(g.tAm, g.sAm, m) : 0;
    }
  } else {
    int64_t m = m0 + a_fix;
    a_okm[0] = m < g.M;
    a_offm[0] = a_okm[0] ? goff(g.tAm, g.sAm, m) : 0;
  }
  if (BKF) {
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      int64_t n = n0 + b_var0 + BSTEP * i;
      b_okn[i] = n < g.N;
      b_offn[i] = b_okn[i] ? goff(g.tBn, g.sBn, n) : 0;
    }
  } else {
    int64_t n = n0 + b_fix;
    b_okn[0] = n < g.N;
    b_offn[0] = b_okn[0] ? goff(g.tBn, g.sBn, n) : 0;
  }

  T ra[NPT], rb[NPT];
  auto load = [&](int64_t k0) {
    if (AK) {
      int64_t k = k0 + a_fix;
      bool okk = k < kend;
      int64_t ok_ = okk ? goff(g.tAk, g.sAk, k) : 0;
#pragma unroll
      for (int i = 0; i < NPT; ++i) ra[i] = (okk && a_okm[i]) ? A[a_offm[i] + ok_] : (T)0;
    } else {
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        int64_t k = k0 + a_var0 + ASTEP * i;
        bool ok = a_okm[0] && k < kend;
        ra[i] = ok ? A[a_offm[0] + goff(g.tAk, g.sAk, k)] : (T)0;
      }
    }
    if (BKF) {
      int64_t k = k0 + b_fix;
      bool okk = k < kend;
      int64_t ok_ = okk ? goff(g.tBk, g.sBk, k) : 0;
#pragma unroll
      for (int i = 0; i < NPT; ++i) rb[i] = (okk && b_okn[i]) ? B[b_offn[i] + ok_] : (T)0;
    } else {
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        int64_t k = k0 + b_var0 + BSTEP * i;
        bool ok = b_okn[0] && k < kend;
        rb[i] = ok ? B[b_offn[0] + goff(g.tBk, g.sBk, k)] : (T)0;
      }
    }
  };

  auto store = [&]() {
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      int am = AK ? a_var0 + ASTEP * i : a_fix;
      int ak = AK ? a_fix : a_var0 + ASTEP * i;
      int bn = BKF ? b_var0 + BSTEP * i : b_fix;
      int bk = BKF ? b_fix : b_var0 + BSTEP * i;
      if constexpr (BF) {
        float xa = (float)ra[i];
        uint16_t ha = f2bf_rne(xa);
        Ah[am * (BKT + PAD) + ak] = ha;
        Al[am * (BKT + PAD) + ak] = f2bf_rne(xa - bf2f(ha));
        float xb = (float)rb[i];
        uint16_t hb = f2bf_rne(xb);
        Bh[bn * (BKT + PAD) + bk] = hb;
        Bl[bn * (BKT + PAD) + bk] = f2bf_rne(xb - bf2f(hb));
      } else {
        As[ak * (BM + PAD) + am] = (CT)ra[i];
        Bs[bk * (BN + PAD) + bn] = (CT)rb[i];
      }
    }
  };

  f4_t acc[WT][WT];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int j = 0; j < WT; ++j) acc[i][j] = f4_t{0, 0, 0, 0};

  const int lr = lane & 15, lg = lane >> 4;
  if (kbeg < kend) load(kbeg);
  for (int64_t k0 = kbeg; k0 < kend; k0 += BKT) {
    __syncthreads();
    store();
    __syncthreads();
    if (k0 + BKT < kend) load(k0 + BKT);
    if constexpr (BF) {
      bf8_t ah[WT], al[WT], bh[WT], bl[WT];
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        int m = wm * WH + i * 16 + lr;
        ah[i] = *(const bf8_t*)&Ah[m * (BKT + PAD) + lg * 8];
        al[i] = *(const bf8_t*)&Al[m * (BKT + PAD) + lg * 8];
        int n = wn * WH + i * 16 + lr;
        bh[i] = *(const bf8_t*)&Bh[n * (BKT + PAD) + lg * 8];
        bl[i] = *(const bf8_t*)&Bl[n * (BKT + PAD) + lg * 8];
      }
#pragma unroll
      for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) {
          if constexpr (BF) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
          }
        }
    } else {
#pragma unroll
      for (int kk = 0; kk < BKT / 4; ++kk) {
        CT a[WT], b[WT];
#pragma unroll
        for (int i = 0; i < WT; ++i) {
          a[i] = As[(kk * 4 + lg) * (BM + PAD) + wm * WH + i * 16 + lr];
          b[i] = Bs[(kk * 4 + lg) * (BN + PAD) + wn * WH + i * 16 + lr];
        }
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
          for (int j = 0; j < WT; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
          }
      }
    }
  }

  gett_epilogue<T>(g, acc, m0, n0, wm, wn, lr, lg);
}

// ---------------------------------------------------------- native kernel
// FP64 storage with FP64 MFMA and FP32 storage with FP32 MFMA. TS x TS
// tile per 256-thread workgroup (2 x 2 waves of TS/2 x TS/2, 16x16x4
// blocks), K staged 16 deep through two LDS buffers with one barrier per
// stage, the loads of two more stages in flight in registers (one in flight:
// 4096^3 FP64 61.3 TFLOP/s, 66.1 now; FP32 125 and 130; a stage of a lone
// 32 x 32 workgroup 0.44 us and 0.27, FP64).
//
// Bound: the matrix pipe, if the loader and the fragment reads stay out of
// its way. A wave issues (TS/32)^2 products per 4 k, 64 (FP64) or 32 (FP32)
// cycles each.
//  - Of an element's offset only the part that changes is recomputed: an
//    operand read along its free index (KF false) takes k from the wave's
//    number, so k's offset (stride or table) is wave-uniform and lives in
//    scalar registers, and the per-lane pointer is fixed for the whole
//    launch; an operand read along k keeps one pointer per row and adds the
//    lane's k offset, which (if it comes from a table) is fetched one stage
//    before the loads that use it. Rows past M or N read the last row
//    instead of being masked (their results are never stored); only the
//    last, partial stage masks k.
//  - Block (i, j) of a wave holds rows WT q + i and columns WT q + j,
//    q < 16, of its sub-tile, so a lane's WT fragments are consecutive in
//    LDS (one 16-byte read for four FP32 or two FP64) and its WT outputs of
//    a row are one vector store.
//
// LDS: [k][m] rows of TS elements, element (k, m) at m ^ sw(k), sw a
// multiple of 4 so that the vectors stay whole; a store of 16 k x 4 m (or
// 8 x 8) by a wave that loads along k then covers every bank evenly.
template <typename T>
__device__ __forceinline__ int native_sw(int k) {
  return std::is_same<T, double>::value ? ((k & 1) << 4) | (((k >> 1) & 3) << 2)
                                        : ((k & 3) << 4) | (((k >> 2) & 3) << 2);
}

// one operand's loader: X(row, k), rows [r0, r0 + TS), TS * BK / 256
// elements per thread and stage
template <typename T, int TS, int BK, bool KF, bool TAB>
struct NativeLoader {
  static constexpr int NPT = TS * BK / 256;
  static constexpr bool UNI = !KF && TS >= 64;   // k uniform over a wave
  static constexpr int STEP = KF ? 256 / BK : 256 / TS;
  static constexpr int MASK = TS < 64 ? TS - 1 : 63;   // swizzle within the row
  static constexpr int NKO = KF ? 1 : NPT;   // k values of a thread in a stage
  const T* p[KF ? NPT : 1];
  const int64_t* tk;         // k offsets from the chunk's first k: table or null
  int64_t sk;                // their stride, if not
  int64_t kn[TAB ? NKO : 1]; // offsets of the next stage's k (!TAB: of its first)
  int kf;                    // KF: k of this thread in a stage; else its first k
  int klen;
  T r[2][NPT];               // two stages in flight

  __device__ __forceinline__ void init(const T* X, int64_t r0, int64_t rows, const int64_t* tr,
                                       int64_t sr, const int64_t* tkk, int64_t skk, int64_t kbeg,
                                       int len) {
    const int t = threadIdx.x;
    const bool tab = TAB && skk < 0;
    tk = tab ? tkk + kbeg : nullptr;
    sk = skk;
    klen = len;
    if (!tab) X += kbeg * skk;
    if constexpr (KF) {
      kf = t % BK;
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        int64_t row = r0 + t / BK + STEP * i;
        row = row < rows ? row : rows - 1;
        p[i] = X + goff(tr, sr, row);
      }
    } else {
      kf = UNI ? __builtin_amdgcn_readfirstlane(t / TS) : t / TS;
      int64_t row = r0 + t % TS;
      row = row < rows ? row : rows - 1;
      p[0] = X + goff(tr, sr, row);
    }
    if constexpr (TAB) offsets(0);
    else kn[0] = kf * sk;
  }
  // kn of the stage at k0, held inside the range (a table ends there)
  __device__ __forceinline__ void offsets(int k0) {
#pragma unroll
    for (int i = 0; i < NKO; ++i) {
      int k = k0 + kf + STEP * i;
      k = k < klen ? k : klen - 1;
      kn[i] = tk ? tk[k] : k * sk;
    }
  }
  // the stage at k0; stages are loaded in order
  __device__ __forceinline__ void load(int k0, int set) {
    if (TAB || k0 + BK <= klen) {
#pragma unroll
      for (int i = 0; i < NPT; ++i)
        r[set][i] = p[KF ? i : 0][KF ? kn[0] : TAB ? kn[TAB ? i % NKO : 0] : kn[0] + (STEP * i) * sk];
    } else {
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        const int k = k0 + kf + (KF ? 0 : STEP * i);
        r[set][i] = k < klen ? p[KF ? i : 0][k * sk] : (T)0;
      }
    }
    if constexpr (TAB) {
      if (k0 + BK > klen) {
#pragma unroll
        for (int i = 0; i < NPT; ++i)
          if (k0 + kf + (KF ? 0 : STEP * i) >= klen) r[set][i] = (T)0;
      }
      offsets(k0 + BK);
    } else {
      kn[0] += BK * sk;
    }
  }
  __device__ __forceinline__ void store(T* s, int set) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const int m = KF ? t / BK + STEP * i : t % TS;
      const int k = KF ? kf : kf + STEP * i;
      s[k * TS + (m ^ (native_sw<T>(k) & MASK))] = r[set][i];
    }
  }
};

// WT consecutive elements, read from LDS in 16-byte pieces (aligned) or
// written to memory (element-aligned)
template <typename T, int WT>
struct NativeVec {
  typedef T vec __attribute__((ext_vector_type(WT)));
  typedef T uvec __attribute__((ext_vector_type(WT), aligned(sizeof(T))));
};

template <typename T, int TS, bool AK, bool BKF, bool TAB>
__global__ __launch_bounds__(256, TS == 128 ? 2 : 4) void gett_native_kernel(GettArgs g) {
  constexpr bool F64 = std::is_same<T, double>::value;
  constexpr int BK = 16, WH = TS / 2, WT = TS / 32, NK = BK / 4;
  constexpr int MASK = TS < 64 ? TS - 1 : 63;
  __shared__ __attribute__((aligned(16))) T smem[2][2][BK * TS];   // [buffer][operand]
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  int64_t tm, tn;
  if (g.band) {
    if (!band_coords(g.tilesM, tm, tn)) return;   // whole workgroup, before any barrier
  } else {
    tile_coords(g.tilesM, g.tilesN, tm, tn);
  }
  const int64_t m0 = tm * TS, n0 = tn * TS;
  const int64_t kbeg = (int64_t)blockIdx.z * g.kchunk;
  const int klen = (int)(kbeg + g.kchunk < g.K ? g.kchunk : g.K - kbeg);

  NativeLoader<T, TS, BK, AK, TAB> la;
  NativeLoader<T, TS, BK, BKF, TAB> lb;
  la.init((const T*)g.A, m0, g.M, g.tAm, g.sAm, g.tAk, g.sAk, kbeg, klen);
  lb.init((const T*)g.B, n0, g.N, g.tBn, g.sBn, g.tBk, g.sBk, kbeg, klen);

  typedef typename std::conditional<F64, d4_t, f4_t>::type acc_t;
  acc_t acc[WT][WT];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int j = 0; j < WT; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  const int lr = lane & 15, lg = lane >> 4;
  const int ma = wm * WH + WT * lr, nb = wn * WH + WT * lr;
  la.load(0, 0);
  lb.load(0, 0);
  if (BK < klen) {
    la.load(BK, 1);
    lb.load(BK, 1);
  }
  la.store(smem[0][0], 0);
  lb.store(smem[0][1], 0);
  if (2 * BK < klen) {
    la.load(2 * BK, 0);
    lb.load(2 * BK, 0);
  }
  __syncthreads();
  // the stage at k0, P = its number mod 2
  auto stage = [&](int k0, auto par) {
    constexpr int P = decltype(par)::value;
    const T* As = smem[P][0];
    const T* Bs = smem[P][1];
    typedef typename NativeVec<T, WT>::vec vec;
    vec a[2], b[2];
    auto frag = [&](int kk) {
      const int k = kk * 4 + lg, sw = native_sw<T>(k) & MASK;
      a[kk & 1] = *(const vec*)(As + k * TS + (ma ^ sw));
      b[kk & 1] = *(const vec*)(Bs + k * TS + (nb ^ sw));
    };
    frag(0);
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      if (kk + 1 < NK) frag(kk + 1);
      if (kk == 1) {
        // the first products are in the matrix pipe: store the next stage
        // (the other buffer was last read before the barrier that ended
        // the previous stage) and start the loads of the one two after it
        __builtin_amdgcn_sched_barrier(0);
        if (k0 + BK < klen) {
          la.store(smem[P ^ 1][0], P ^ 1);
          lb.store(smem[P ^ 1][1], P ^ 1);
          if (k0 + 3 * BK < klen) {
            la.load(k0 + 3 * BK, P ^ 1);
            lb.load(k0 + 3 * BK, P ^ 1);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) {
          if constexpr (F64)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kk & 1][i], b[kk & 1][j],
                                                             acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[kk & 1][i], b[kk & 1][j],
                                                             acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  };
  for (int k0 = 0; k0 < klen; k0 += 2 * BK) {
    stage(k0, std::integral_constant<int, 0>());
    if (k0 + BK < klen) stage(k0 + BK, std::integral_constant<int, 1>());
  }

  // lane holds D[q][lr] of each block, q = 4 lg + r (FP32) or 4 r + lg
  // (FP64): rows m0 + wm WH + WT q + i, columns n .. n + WT - 1
  const int64_t n = n0 + wn * WH + WT * lr;
  const int64_t mb = m0 + wm * WH;
  if (n >= g.N) return;
  const int nw = g.N - n < WT ? (int)(g.N - n) : WT;   // live columns of this lane
  typedef typename NativeVec<T, WT>::uvec uvec;
  if (g.partial || (g.sCn == 1 && g.sCm >= 0)) {
    T* P = g.partial ? (T*)g.partial + (int64_t)blockIdx.z * g.M * g.N : (T*)g.C;
    const int64_t ld = g.partial ? g.N : g.sCm;
    const double al = g.partial ? 1.0 : g.alpha, be = g.partial ? 0.0 : g.beta;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        const int64_t m = mb + WT * (F64 ? 4 * r + lg : 4 * lg + r) + i;
        if (m >= g.M) continue;
        T* c = P + m * ld + n;
        if (nw == WT) {
          uvec v;
          if (be != 0.0) {
            const uvec o = *(const uvec*)c;
#pragma unroll
            for (int j = 0; j < WT; ++j) v[j] = (T)(al * (double)acc[i][j][r] + be * (double)o[j]);
          } else {
#pragma unroll
            for (int j = 0; j < WT; ++j) v[j] = (T)(al * (double)acc[i][j][r]);
          }
          *(uvec*)c = v;
        } else {
#pragma unroll
          for (int j = 0; j < WT; ++j)
            if (j < nw) {
              double v = al * (double)acc[i][j][r];
              if (be != 0.0) v += be * (double)c[j];
              c[j] = (T)v;
            }
        }
      }
    return;
  }
  T* C = (T*)g.C;
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    if (j >= nw) continue;
    const int64_t on = goff(g.tCn, g.sCn, n + j);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        const int64_t m = mb + WT * (F64 ? 4 * r + lg : 4 * lg + r) + i;
        if (m >= g.M) continue;
        const int64_t o = on + goff(g.tCm, g.sCm, m);
        double v = g.alpha * (double)acc[i][j][r];
        if (g.beta != 0.0) v += g.beta * (double)C[o];
        C[o] = (T)v;
      }
  }
}

// split-K reduction + epilogue. A block takes 64 (or, with few partials, 256)
// consecutive outputs; ZW waves share an output's partials (z = wave mod ZW,
// eight loads in flight each) and meet in LDS in a fixed order. One thread
// per output, walking the partials, was latency-bound: 12.7 us for 64 of
// 256 x 256 FP32, 3.6 now.
template <typename T, typename CT, int ZW>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GettArgs g, int nsplit) {
  constexpr int EB = 256 / ZW;   // outputs per block and turn
  __shared__ double sh[ZW][EB];
  const int64_t MN = g.M * g.N;
  const CT* __restrict__ P = (const CT*)g.partial;
  T* C = (T*)g.C;
  const int ei = threadIdx.x % EB, zi = threadIdx.x / EB;
  for (int64_t e0 = blockIdx.x * (int64_t)EB; e0 < MN; e0 += (int64_t)gridDim.x * EB) {
    const int64_t e = e0 + ei;
    double s = 0.0;
    if (e < MN) {
      const CT* p = P + e;
      int z = zi;
      for (; z + 7 * ZW < nsplit; z += 8 * ZW) {
        CT v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = p[(int64_t)(z + q * ZW) * MN];
#pragma unroll
        for (int q = 0; q < 8; ++q) s += (double)v[q];
      }
      for (; z < nsplit; z += ZW) s += (double)p[(int64_t)z * MN];
    }
    if constexpr (ZW > 1) {
      __syncthreads();
      sh[zi][ei] = s;
      __syncthreads();
      if (zi != 0) continue;
      s = sh[0][ei];
#pragma unroll
      for (int q = 1; q < ZW; ++q) s += sh[q][ei];
    }
    if (e >= MN) continue;
    const int64_t n = e % g.N, m = e / g.N;
    const int64_t o = goff(g.tCm, g.sCm, m) + goff(g.tCn, g.sCn, n);
    double v = g.alpha * s;
    if (g.beta != 0.0) v += g.beta * (double)C[o];
    C[o] = (T)v;
  }
}

template <typename T, typename CT>
static void splitk_reduce(itg_ctx* ctx, const GettArgs& g, int nsplit) {
  const int64_t MN = g.M * g.N;
  if (nsplit >= 8)
    splitk_reduce_kernel<T, CT, 4><<<itg_blocks(MN, 64, 8192), 256, 0, ctx->stream>>>(g, nsplit);
  else
    splitk_reduce_kernel<T, CT, 1><<<itg_blocks(MN, 256, 4096), 256, 0, ctx->stream>>>(g, nsplit);
}

// Contractions with at most 16 outputs (scalars, short vectors; dot-like):
// every block reduces a K-range for all outputs in FP64, then one reduction.
template <typename T>
__global__ __launch_bounds__(256) void small_out_kernel(GettArgs g, double* part) {
  const T* A = (const T*)g.A;
  const T* B = (const T*)g.B;
  int mn = (int)(g.M * g.N);
  double acc[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.0;
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < g.K;
       k += (int64_t)gridDim.x * blockDim.x) {
    int64_t ak = goff(g.tAk, g.sAk, k), bk = goff(g.tBk, g.sBk, k);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if (e < mn) {
        int64_t m = e % g.M, n = e / g.M;
        acc[e] += (double)A[goff(g.tAm, g.sAm, m) + ak] * (double)B[bk + goff(g.tBn, g.sBn, n)];
      }
    }
  }
  __shared__ double sh[4][16];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    double v = acc[e];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) sh[w][e] = v;
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    int e = threadIdx.x;
    part[blockIdx.x * 16 + e] = sh[0][e] + sh[1][e] + sh[2][e] + sh[3][e];
  }
}

template <typename T>
__global__ void small_out_finish(GettArgs g, const double* part, int nblk) {
  int e = threadIdx.x;
  int mn = (int)(g.M * g.N);
  if (e >= mn) return;
  double s = 0.0;
  for (int b = 0; b < nblk; ++b) s += part[b * 16 + e];
  int64_t m = e % g.M, n = e / g.M;
  T* C = (T*)g.C;
  int64_t o = goff(g.tCm, g.sCm, m) + goff(g.tCn, g.sCn, n);
  double v = g.alpha * s;
  if (g.beta != 0.0) v += g.beta * (double)C[o];
  C[o] = (T)v;
}

// ======================================================================
// host side: plans
// A contraction with one small operand: the big operand X carries the free
// modes F (at most 3) and the summed modes K, the small one Y the free modes
// G and K, with K and G small (K <= 64, G <= 32, K G <= 1024). It streams X
// once through sic_kernel, which forms every offset from the modes' extents
// and strides: no offset tables (which for a non-mergeable F would have F
// entries, built on the host for every new shape).
constexpr int SIC_KMAX = 64, SIC_GMAX = 32;
constexpr int64_t SIC_FMIN = 4096;   // smaller F: the GEMM kernel is fine
struct SicArgs {
  const void* X;
  const void* Y;
  void* C;
  int64_t F;
  int nf, ng, nk, G, K;
  int64_t fd[3], fx[3], fc[3];   // F: extent, stride in X, stride in C
  int64_t gd[4], gy[4], gc[4];   // G: extent, stride in Y, stride in C
  int64_t kd[4], kx[4], ky[4];   // K: extent, stride in X, stride in Y
  double alpha, beta;
};

struct itg_plan {
  int64_t M = 1, N = 1, K = 1;
  bool swap = false;
  int64_t sAm = 0, sAk = 0, sBk = 0, sBn = 0, sCm = 0, sCn = 0;
  int64_t* dtab = nullptr;   // device tables (concatenated)
  int64_t oAm = -1, oAk = -1, oBk = -1, oBn = -1, oCm = -1, oCn = -1;  // offsets into dtab
  bool akfast = false, bkfast = false;
  size_t bytes = 0;
  // small-operand form (no tables): X is the A-role operand if sic_xa
  bool sic = false, sic_xa = true;
  SicArgs sa = {};
};

// blockIdx.y takes GM of the G outputs (its own part of Y in LDS), so that a
// small F still fills the chip; X is then read once per part, from L2.
// F = 305000, K = G = 8 FP64: 24 us with 64-bit index arithmetic and every
// output in one thread, 19 now; the operator products of a DMRG sweep on a
// 4 x 6 cylinder take 8.6 us on average.
template <typename T, int GM, typename I>
__global__ __launch_bounds__(256) void sic_kernel(SicArgs a) {
  __shared__ T ys[SIC_KMAX * GM];      // Y(k, g0 + g) at k GM + g
  __shared__ int64_t kox[SIC_KMAX];    // offset of k in X
  __shared__ int64_t goc[GM];          // offset of g0 + g in C
  const int t = threadIdx.x;
  const int g0 = (int)blockIdx.y * GM, ng = min(GM, a.G - g0);
  const T* __restrict__ Y = (const T*)a.Y;
  for (int e = t; e < a.K * GM; e += 256) {
    int rk = e / GM, rg = g0 + e % GM;
    int64_t o = 0;
    const bool live = e % GM < ng;
    for (int q = 0; q < a.nk; ++q) { o += (rk % (int)a.kd[q]) * a.ky[q]; rk /= (int)a.kd[q]; }
    for (int q = 0; q < a.ng; ++q) { o += (rg % (int)a.gd[q]) * a.gy[q]; rg /= (int)a.gd[q]; }
    ys[e] = live ? Y[o] : (T)0;
  }
  for (int k = t; k < a.K; k += 256) {
    int r = k;
    int64_t o = 0;
    for (int q = 0; q < a.nk; ++q) { o += (r % (int)a.kd[q]) * a.kx[q]; r /= (int)a.kd[q]; }
    kox[k] = o;
  }
  for (int g = t; g < ng; g += 256) {
    int r = g0 + g;
    int64_t o = 0;
    for (int q = 0; q < a.ng; ++q) { o += (r % (int)a.gd[q]) * a.gc[q]; r /= (int)a.gd[q]; }
    goc[g] = o;
  }
  __syncthreads();
  const int64_t f = (int64_t)blockIdx.x * 256 + t;
  if (f >= a.F) return;
  int64_t ox = 0, oc = 0;
  I r = (I)f;
  for (int q = 0; q < a.nf; ++q) {
    const I dq = (I)a.fd[q], rq = r / dq, i = r - rq * dq;
    r = rq;
    ox += (int64_t)i * a.fx[q];
    oc += (int64_t)i * a.fc[q];
  }
  const T* __restrict__ X = (const T*)a.X + ox;
  T acc[GM];
#pragma unroll
  for (int g = 0; g < GM; ++g) acc[g] = (T)0;
  int k = 0;
  for (; k + 8 <= a.K; k += 8) {
    T xv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) xv[q] = X[kox[k + q]];
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int g = 0; g < GM; ++g) acc[g] += xv[q] * ys[(k + q) * GM + g];
  }
  for (; k < a.K; ++k) {
    const T xv = X[kox[k]];
#pragma unroll
    for (int g = 0; g < GM; ++g) acc[g] += xv * ys[k * GM + g];
  }
  T* __restrict__ C = (T*)a.C + oc;
#pragma unroll
  for (int g = 0; g < GM; ++g) {
    if (g < ng) {
      T v = (T)a.alpha * acc[g];
      if (a.beta != 0.0) v += (T)a.beta * C[goc[g]];
      C[goc[g]] = v;
    }
  }
}

template <typename T>
static void launch_sic_t(itg_ctx* ctx, const SicArgs& a, unsigned nblk) {
  // outputs per thread: all of them for a large F, fewer until the grid has
  // four workgroups per CU
  int gm = a.G <= 4 ? 4 : a.G <= 8 ? 8 : a.G <= 16 ? 16 : 32;
  const int64_t want = 4 * (int64_t)std::max(ctx->num_cu, 1);
  while (gm > 4 && (int64_t)nblk * ((a.G + gm - 1) / gm) < want) gm /= 2;
  const dim3 grid(nblk, (a.G + gm - 1) / gm);
  auto go = [&](auto kernel) { kernel<<<grid, 256, 0, ctx->stream>>>(a); };
  if (a.F <= 0x7fffffff) {
    if (gm == 4) go(sic_kernel<T, 4, uint32_t>);
    else if (gm == 8) go(sic_kernel<T, 8, uint32_t>);
    else if (gm == 16) go(sic_kernel<T, 16, uint32_t>);
    else go(sic_kernel<T, SIC_GMAX, uint32_t>);
  } else {
    go(sic_kernel<T, SIC_GMAX, int64_t>);
  }
}

static int launch_sic(itg_ctx* ctx, int dtype, const itg_plan* p, const void* A, const void* B,
                      void* C, double alpha, double beta) {
  SicArgs a = p->sa;
  a.X = p->sic_xa ? A : B;
  a.Y = p->sic_xa ? B : A;
  a.C = C;
  a.alpha = alpha;
  a.beta = beta;
  const int64_t nblk = (a.F + 255) / 256;
  if (nblk > 0x7fffffff) return itg_fail(ctx, ITG_EUNSUPPORTED, "contraction too large");
  const int tk = itg_tstart(ctx, ITG_K_GETT);
  if (dtype == ITG_F64) launch_sic_t<double>(ctx, a, (unsigned)nblk);
  else launch_sic_t<float>(ctx, a, (unsigned)nblk);
  ITG_LAUNCH_CHECK(ctx);
  const double es = dtype == ITG_F64 ? 8.0 : 4.0;
  itg_tstop(ctx, tk, ITG_K_GETT, 2.0 * a.F * a.G * a.K,
            es * (a.F * a.K + a.F * a.G * (beta != 0.0 ? 2 : 1)));
  return ITG_OK;
}

void itg_plan_cache_clear(itg_ctx* ctx) {
  for (auto& kv : ctx->plans) {
    if (kv.second->dtab) hipFree(kv.second->dtab);
    delete kv.second;
  }
  ctx->plans.clear();
  ctx->plan_bytes = 0;
}

namespace {
struct Mode {
  int64_t d;
  int64_t s1, s2;  // strides in the two tensors that carry this mode
};

// order by s1 ascending and merge modes that are contiguous continuations in
// both tensors
std::vector<Mode> canon(std::vector<Mode> v, bool by_second) {
  std::vector<Mode> w;
  for (auto& x : v)
    if (x.d != 1) w.push_back(x);
  std::stable_sort(w.begin(), w.end(), [&](const Mode& a, const Mode& b) {
    return by_second ? a.s2 < b.s2 : a.s1 < b.s1;
  });
  std::vector<Mode> out;
  for (auto& x : w) {
    if (!out.empty() && out.back().s1 * out.back().d == x.s1 &&
        out.back().s2 * out.back().d == x.s2) {
      out.back().d *= x.d;
    } else {
      out.push_back(x);
    }
  }
  return out;
}

// offsets of a group for tensor `which` (1 or 2); returns stride or -1 with table
int64_t group_offsets(const std::vector<Mode>& g, int which, std::vector<int64_t>& tab) {
  if (g.empty()) return 0;
  if (g.size() == 1) return which == 1 ? g[0].s1 : g[0].s2;
  int64_t n = 1;
  for (auto& x : g) n *= x.d;
  tab.resize(n);
  for (int64_t i = 0; i < n; ++i) {
    int64_t rem = i, o = 0;
    for (auto& x : g) {
      int64_t j = rem % x.d;
      rem /= x.d;
      o += j * (which == 1 ? x.s1 : x.s2);
    }
    tab[i] = o;
  }
  return -1;
}
}  // namespace

static int build_plan(itg_ctx* ctx, const std::string& key, int rA, const int64_t* dA,
                      const int32_t* lA, int rB, const int64_t* dB, const int32_t* lB, int rC,
                      const int64_t* dC, const int32_t* lC, itg_plan** out) {
  // strides
  int64_t sA[ITG_MAX_RANK], sB[ITG_MAX_RANK], sC[ITG_MAX_RANK];
  int64_t s = 1;
  for (int i = 0; i < rA; ++i) { sA[i] = s; s *= dA[i]; }
  s = 1;
  for (int i = 0; i < rB; ++i) { sB[i] = s; s *= dB[i]; }
  s = 1;
  for (int i = 0; i < rC; ++i) { sC[i] = s; s *= dC[i]; }
  auto find = [](const int32_t* l, int r, int32_t x) {
    for (int i = 0; i < r; ++i) if (l[i] == x) return i;
    return -1;
  };
  // C's fastest non-unit mode decides the operand roles: it must be an n-mode
  bool swap = false;
  for (int i = 0; i < rC; ++i) {
    if (dC[i] == 1) continue;
    swap = find(lA, rA, lC[i]) >= 0;
    break;
  }
  const int32_t *la = lA, *lb = lB;
  const int64_t *da = dA, *db = dB, *psA = sA, *psB = sB;
  int ra = rA, rb = rB;
  if (swap) {
    std::swap(la, lb); std::swap(da, db); std::swap(psA, psB); std::swap(ra, rb);
  }
  std::vector<Mode> gm, gn, gk;
  for (int i = 0; i < ra; ++i) {
    int jb = find(lb, rb, la[i]);
    if (jb >= 0) {
      gk.push_back({da[i], psA[i], psB[jb]});
    } else {
      int jc = find(lC, rC, la[i]);
      gm.push_back({da[i], psA[i], sC[jc]});
    }
  }
  for (int i = 0; i < rb; ++i) {
    if (find(la, ra, lb[i]) >= 0) continue;
    int jc = find(lC, rC, lb[i]);
    gn.push_back({db[i], psB[i], sC[jc]});
  }
  // K order: by A's strides if A's unit-stride mode is contracted, else by B's
  bool a_unit_in_k = false, b_unit_in_k = false;
  for (auto& x : gk) {
    if (x.d > 1 && x.s1 == 1) a_unit_in_k = true;
    if (x.d > 1 && x.s2 == 1) b_unit_in_k = true;
  }
  std::vector<Mode> cm = canon(gm, false), cn = canon(gn, false);
  std::vector<Mode> ck = canon(gk, !a_unit_in_k && b_unit_in_k);
  itg_plan* p = new itg_plan();
  p->swap = swap;
  for (auto& x : cm) p->M *= x.d;
  for (auto& x : cn) p->N *= x.d;
  for (auto& x : ck) p->K *= x.d;
  // the small-operand form: the big free group of at most 3 modes, the
  // other free group and K small
  if (ck.size() <= 4 && p->K <= SIC_KMAX) {
    const bool xa = cm.size() <= 3 && cn.size() <= 4 && p->N <= SIC_GMAX &&
                    p->N * p->K <= SIC_KMAX * SIC_GMAX && p->M >= SIC_FMIN;
    const bool xb = !xa && cn.size() <= 3 && cm.size() <= 4 && p->M <= SIC_GMAX &&
                    p->M * p->K <= SIC_KMAX * SIC_GMAX && p->N >= SIC_FMIN;
    if (xa || xb) {
      // Mode strides: M {A, C}, N {B, C}, K {A, B}
      const std::vector<Mode>& F = xa ? cm : cn;
      const std::vector<Mode>& G = xa ? cn : cm;
      SicArgs& a = p->sa;
      a.F = xa ? p->M : p->N;
      a.G = (int)(xa ? p->N : p->M);
      a.K = (int)p->K;
      a.nf = (int)F.size();
      a.ng = (int)G.size();
      a.nk = (int)ck.size();
      for (int q = 0; q < a.nf; ++q) { a.fd[q] = F[q].d; a.fx[q] = F[q].s1; a.fc[q] = F[q].s2; }
      for (int q = 0; q < a.ng; ++q) { a.gd[q] = G[q].d; a.gy[q] = G[q].s1; a.gc[q] = G[q].s2; }
      for (int q = 0; q < a.nk; ++q) {
        a.kd[q] = ck[q].d;
        a.kx[q] = xa ? ck[q].s1 : ck[q].s2;
        a.ky[q] = xa ? ck[q].s2 : ck[q].s1;
      }
      p->sic = true;
      p->sic_xa = xa;
      if (ctx->plans.size() > 4096) {
        hipStreamSynchronize(ctx->stream);
        itg_plan_cache_clear(ctx);
      }
      ctx->plans[key] = p;
      *out = p;
      return ITG_OK;
    }
  }
  std::vector<int64_t> tAm, tAk, tBk, tBn, tCm, tCn;
  p->sAm = group_offsets(cm, 1, tAm);
  p->sCm = group_offsets(cm, 2, tCm);
  p->sBn = group_offsets(cn, 1, tBn);
  p->sCn = group_offsets(cn, 2, tCn);
  p->sAk = group_offsets(ck, 1, tAk);
  p->sBk = group_offsets(ck, 2, tBk);
  // load directions: contiguous along the free index if its first mode has
  // unit stride, else along k if k's first mode has unit stride
  p->akfast = !(!cm.empty() && cm[0].s1 == 1) && (!ck.empty() && ck[0].s1 == 1);
  p->bkfast = !(!cn.empty() && cn[0].s1 == 1) && (!ck.empty() && ck[0].s2 == 1);
  size_t total = tAm.size() + tAk.size() + tBk.size() + tBn.size() + tCm.size() + tCn.size();
  if (total) {
    std::vector<int64_t> all;
    all.reserve(total);
    auto put = [&](std::vector<int64_t>& v, int64_t& o) {
      if (!v.empty()) { o = (int64_t)all.size(); all.insert(all.end(), v.begin(), v.end()); }
    };
    put(tAm, p->oAm); put(tAk, p->oAk); put(tBk, p->oBk);
    put(tBn, p->oBn); put(tCm, p->oCm); put(tCn, p->oCn);
    if (hipMalloc(&p->dtab, total * sizeof(int64_t)) != hipSuccess) {
      delete p;
      return itg_fail(ctx, ITG_EOOM, "plan table allocation failed");
    }
    hipError_t e = hipMemcpyAsync(p->dtab, all.data(), total * sizeof(int64_t),
                                  hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
      hipFree(p->dtab);
      delete p;
      return itg_fail(ctx, ITG_EHIP, "plan upload failed: %s", hipGetErrorString(e));
    }
    p->bytes = total * sizeof(int64_t);
  }
  // bound the cache
  if (ctx->plans.size() > 4096 || ctx->plan_bytes + p->bytes > ((size_t)1 << 30)) {
    hipStreamSynchronize(ctx->stream);
    itg_plan_cache_clear(ctx);
  }
  ctx->plans[key] = p;
  ctx->plan_bytes += p->bytes;
  *out = p;
  return ITG_OK;
}

template <typename T, int MODE>
static int launch_gett_t(itg_ctx* ctx, GettArgs& g, bool ak, bool bk) {
  using TR = GettTraits<MODE>;
  using CT = float;
  g.tilesM = (g.M + TR::BM - 1) / TR::BM;
  g.tilesN = (g.N + TR::BN - 1) / TR::BN;
  int64_t tiles = g.tilesM * g.tilesN;
  if (tiles > 0x7fffffff) return itg_fail(ctx, ITG_EUNSUPPORTED, "contraction too large");
  // split K when the output has too few tiles to fill the chip
  int nsplit = 1;
  int64_t target = 2 * (int64_t)std::max(ctx->num_cu, 1);
  if (!g.band && tiles < target && g.K >= TR::BKT * 16) {
    // at least 4 k-tiles per split
    int64_t want = (target + tiles - 1) / tiles;
    int64_t maxs = g.K / (TR::BKT * 4);
    nsplit = (int)std::max<int64_t>(1, std::min<int64_t>({want, maxs, 64}));
  }
  if (nsplit > 1 && ctx->fixed_ws) {
    // a no-alloc call: no more splits than its fixed scratch holds
    const size_t per = (size_t)g.M * g.N * sizeof(CT);
    nsplit = (int)std::max<size_t>(1, std::min<size_t>((size_t)nsplit, ctx->fixed_ws_bytes / per));
  }
  g.partial = nullptr;
  g.kchunk = g.K;
  if (nsplit > 1) {
    int64_t chunk = (g.K + nsplit - 1) / nsplit;
    chunk = (chunk + TR::BKT - 1) / TR::BKT * TR::BKT;
    nsplit = (int)((g.K + chunk - 1) / chunk);
    g.kchunk = chunk;
    void* ws;
    if (ctx->fixed_ws) {
      ws = ctx->fixed_ws;
    } else {
      int rc = itg_workspace(ctx, (size_t)nsplit * g.M * g.N * sizeof(CT), &ws);
      if (rc) return rc;
    }
    g.partial = ws;
  }
  dim3 grid((unsigned)tiles, 1, (unsigned)nsplit);
  int tk = itg_tstart(ctx, ITG_K_GETT);
  if (ak && bk) gett_kernel<T, MODE, true, true><<<grid, 256, 0, ctx->stream>>>(g);
  else if (ak) gett_kernel<T, MODE, true, false><<<grid, 256, 0, ctx->stream>>>(g);
  else if (bk) gett_kernel<T, MODE, false, true><<<grid, 256, 0, ctx->stream>>>(g);
  else gett_kernel<T, MODE, false, false><<<grid, 256, 0, ctx->stream>>>(g);
  ITG_LAUNCH_CHECK(ctx);
  itg_tstop(ctx, tk, ITG_K_GETT, 2.0 * g.M * g.N * g.K,
            (double)sizeof(T) * (g.M * g.K + g.K * g.N + g.M * g.N * (g.beta != 0.0 ? 2 : 1)));
  if (nsplit > 1) {
    splitk_reduce<T, CT>(ctx, g, nsplit);
    ITG_LAUNCH_CHECK(ctx);
  }
  return ITG_OK;
}

template <typename T, int TS, bool TAB>
static void native_kernel(itg_ctx* ctx, const GettArgs& g, dim3 grid, bool ak, bool bk) {
  hipStream_t st = ctx->stream;
  if (ak && bk) gett_native_kernel<T, TS, true, true, TAB><<<grid, 256, 0, st>>>(g);
  else if (ak) gett_native_kernel<T, TS, true, false, TAB><<<grid, 256, 0, st>>>(g);
  else if (bk) gett_native_kernel<T, TS, false, true, TAB><<<grid, 256, 0, st>>>(g);
  else gett_native_kernel<T, TS, false, false, TAB><<<grid, 256, 0, st>>>(g);
}

template <typename T, int TS>
static void native_kernel(itg_ctx* ctx, const GettArgs& g, dim3 grid, bool ak, bool bk) {
  if (g.sAk < 0 || g.sBk < 0) native_kernel<T, TS, true>(ctx, g, grid, ak, bk);
  else native_kernel<T, TS, false>(ctx, g, grid, ak, bk);
}

// Tile and K split of the native kernel by estimated time. A CU with nw
// workgroups takes lat + (nw - 1) mf per 16-deep stage: lat is the stage
// of a workgroup alone on its CU (barrier, LDS and load latency exposed), mf
// what each further one adds; a split adds a launch and its partials'
// traffic. Measured on MI355X (us; one workgroup per CU and many):
//            FP64 lat  mf      FP32 lat  mf
//   32 x 32       0.27 0.175        0.21 0.108
//   64 x 64       0.77 0.50         0.41 0.315
// 128 x 128          -    -         1.23 1.05
// FP64 at 128 x 128 gains nothing over 64 x 64 (59 against 61 TFLOP/s at
// 4096^3: 64 cycles per product hide the smaller tile's reads) and rounds
// worse, so it is not built. The estimates are within 15% of the measured
// times over 26 shapes, 80 x 20 x 100 to 4096 x 4096 x 1024, and on nearly all of
// them pick the fastest tile and split or one within 10% of it.
struct NativeChoice {
  int ts, nsplit;
};
static NativeChoice choose_native(const itg_ctx* ctx, const GettArgs& g, bool f64) {
  struct Tile {
    int ts;
    double lat, mf;
  };
  static const Tile t64[] = {{32, 0.27, 0.175}, {64, 0.77, 0.50}};
  static const Tile t32[] = {{32, 0.21, 0.108}, {64, 0.41, 0.315}, {128, 1.23, 1.05}};
  const Tile* tiles = f64 ? t64 : t32;
  const int nt = f64 ? 2 : 3;
  const double cus = std::max(ctx->num_cu, 1);
  const double es = f64 ? 8.0 : 4.0;
  const double mn = (double)g.M * (double)g.N;
  NativeChoice best = {64, 1};
  double tbest = -1.0;
  for (int i = 0; i < nt; ++i) {
    const int ts = tiles[i].ts;
    // a band of one tile above the diagonal has to hold 64 of them
    if (g.band && ts < 64) continue;
    const double nm = (double)((g.M + ts - 1) / ts), nn = (double)((g.N + ts - 1) / ts);
    const double wg = g.band ? 0.5 * nm * (nn + 3.0) : nm * nn;
    for (int sp = 1; sp <= 64; sp *= 2) {
      if (sp > 1 && (g.band || g.K < 32 * (int64_t)sp)) break;
      // no more partials than a no-alloc call's scratch holds
      if (sp > 1 && ctx->fixed_ws && mn * es * sp > (double)ctx->fixed_ws_bytes) break;
      const double nw = std::ceil(wg * sp / cus);
      const double stages = std::ceil(std::ceil((double)g.K / sp) / 16.0);
      double t = stages * (tiles[i].lat + (nw - 1.0) * tiles[i].mf);
      if (sp > 1) t += 2.5 + (sp + 1.0) * mn * es / 3.0e6;
      if (tbest < 0.0 || t < tbest) {
        tbest = t;
        best = {ts, sp};
      }
    }
  }
  return best;
}

template <typename T>
static int launch_native(itg_ctx* ctx, GettArgs& g, bool ak, bool bk) {
  constexpr bool F64 = std::is_same<T, double>::value;
  NativeChoice c = choose_native(ctx, g, F64);
  g.tilesM = (g.M + c.ts - 1) / c.ts;
  g.tilesN = (g.N + c.ts - 1) / c.ts;
  const int64_t tiles = g.band ? (band_tiles(g.tilesM) + 7) / 8 * 8 : g.tilesM * g.tilesN;
  if (tiles > 0x7fffffff) return itg_fail(ctx, ITG_EUNSUPPORTED, "contraction too large");
  // a workgroup counts its k in 32 bits
  constexpr int64_t kMaxChunk = (int64_t)1 << 30;
  int64_t nsplit = std::max<int64_t>(c.nsplit, (g.K + kMaxChunk - 1) / kMaxChunk);
  g.partial = nullptr;
  g.kchunk = g.K;
  if (nsplit > 1) {
    const int64_t chunk = ((g.K + nsplit - 1) / nsplit + 15) / 16 * 16;
    nsplit = (g.K + chunk - 1) / chunk;
    g.kchunk = chunk;
    void* ws = ctx->fixed_ws;
    if (!ws) {
      int rc = itg_workspace(ctx, (size_t)nsplit * g.M * g.N * sizeof(T), &ws);
      if (rc) return rc;
    }
    g.partial = ws;
  }
  dim3 grid((unsigned)tiles, 1, (unsigned)nsplit);
  const int tk = itg_tstart(ctx, ITG_K_GETT);
  if (c.ts == 32) native_kernel<T, 32>(ctx, g, grid, ak, bk);
  else if (F64 || c.ts == 64) native_kernel<T, 64>(ctx, g, grid, ak, bk);
  else native_kernel<float, 128>(ctx, g, grid, ak, bk);
  ITG_LAUNCH_CHECK(ctx);
  itg_tstop(ctx, tk, ITG_K_GETT, 2.0 * g.M * g.N * g.K,
            (double)sizeof(T) * (g.M * g.K + g.K * g.N + g.M * g.N * (g.beta != 0.0 ? 2 : 1)));
  if (nsplit > 1) {
    splitk_reduce<T, T>(ctx, g, (int)nsplit);
    ITG_LAUNCH_CHECK(ctx);
  }
  return ITG_OK;
}

static int launch_gett(itg_ctx* ctx, int dtype, int mode, GettArgs& g, bool ak, bool bk) {
  if (g.M * g.N <= 16) {
    int nblk = (int)std::min<int64_t>(std::max<int64_t>((g.K + 255) / 256, 1), 512);
    double* part = ctx->red + 64;
    if (dtype == ITG_F64) {
      small_out_kernel<double><<<nblk, 256, 0, ctx->stream>>>(g, part);
      small_out_finish<double><<<1, 64, 0, ctx->stream>>>(g, part, nblk);
    } else {
      small_out_kernel<float><<<nblk, 256, 0, ctx->stream>>>(g, part);
      small_out_finish<float><<<1, 64, 0, ctx->stream>>>(g, part, nblk);
    }
    ITG_LAUNCH_CHECK(ctx);
    return ITG_OK;
  }
  if (dtype == ITG_F64) {
    if (mode == ITG_MODE_NATIVE) return launch_native<double>(ctx, g, ak, bk);
    if (mode == ITG_MODE_F32) return launch_gett_t<double, ITG_MODE_F32>(ctx, g, ak, bk);
    return launch_gett_t<double, ITG_MODE_BF16X3>(ctx, g, ak, bk);
  }
  if (mode == ITG_MODE_BF16X3) return launch_gett_t<float, ITG_MODE_BF16X3>(ctx, g, ak, bk);
  return launch_native<float>(ctx, g, ak, bk);
}

// C(r, c) = C(c, r) for r < c from the lower triangle, through 32 x 32 LDS
// tiles (block (bi, bj) writes the upper tile at rows bi, columns bj >= bi)
template <typename T>
__global__ __launch_bounds__(256) void mirror_lower_kernel(int64_t n, T* __restrict__ C,
                                                           int64_t ldc) {
  __shared__ T t[32][33];
  const int64_t bi = blockIdx.x, bj = blockIdx.y;
  if (bj < bi) return;
  for (int yy = threadIdx.y; yy < 32; yy += 8) {
    int64_t r = bj * 32 + threadIdx.x, c = bi * 32 + yy;
    if (r < n && c < n) t[yy][threadIdx.x] = C[r + c * ldc];
  }
  __syncthreads();
  for (int yy = threadIdx.y; yy < 32; yy += 8) {
    int64_t r = bi * 32 + threadIdx.x, c = bj * 32 + yy;
    if (r < n && c < n && r < c) C[r + c * ldc] = t[threadIdx.x][yy];
  }
}

static int mirror_lower(itg_ctx* ctx, int dtype, int64_t n, void* C, int64_t ldc) {
  dim3 grid((unsigned)((n + 31) / 32), (unsigned)((n + 31) / 32));
  if (dtype == ITG_F64)
    mirror_lower_kernel<double><<<grid, dim3(32, 8), 0, ctx->stream>>>(n, (double*)C, ldc);
  else
    mirror_lower_kernel<float><<<grid, dim3(32, 8), 0, ctx->stream>>>(n, (float*)C, ldc);
  ITG_LAUNCH_CHECK(ctx);
  return ITG_OK;
}

// Whether C = alpha A A^T (n x n) is computed as its lower triangle (and one
// tile band), mirrored: a band with fewer 64 x 64 tiles than CUs is no faster
// than the whole product, which can split K. FP64, us, band against whole:
// 1024 x 1024: 58 / 59, 512 x 2048: 103 / 39, 256 x 256: 20 / 12; on the other
// side 1500 x 1500: 121 / 150, 2048 x 2048: 220 / 255, 4096 x 4096: 1240 / 1820.
// FP32: 640 x 2048: 66 / 38, 1024 x 512: 24 / 24, 1024 x 2048: 67 / 60; on the other
// side 1400 x 512: 32 / 32, 1500 x 2048: 92 / 120, 4096 x 4096: 769 / 1161 (1200 x
// 512, just below the line, 25 / 31).
static bool band_wins(const itg_ctx* ctx, int mode, int64_t n) {
  return mode != ITG_MODE_NATIVE || band_tiles((n + 63) / 64) >= std::max(ctx->num_cu, 1);
}

// A contraction whose M, N and K modes each merge into one stride is a plain
// product C(m, n) = alpha sum_k A(m, k) B(k, n) + beta C(m, n), elements at
// m sAm + k sAk, k sBk + n sBn, m sCm + n sCn. It runs as a column-major
// GEMM (the vendor library's) when each matrix has a unit stride on one
// side: X(r, c) at r sr + c sc is op 'N' with ld = sc when sr = 1, op 'T'
// with ld = sr when sc = 1. If C's unit stride is along n, C^T = B^T A^T is
// computed instead. Returns 1 for a layout that is not of this kind.
static int contract_on_lib(itg_ctx* ctx, const GettArgs& g) {
  auto as_col = [](int64_t rows, int64_t cols, int64_t sr, int64_t sc, char& op,
                   int64_t& ld) -> bool {
    if ((rows == 1 || sr == 1) && (cols == 1 || sc >= rows)) {
      op = 'N';
      ld = cols == 1 ? rows : sc;
      return true;
    }
    if ((cols == 1 || sc == 1) && (rows == 1 || sr >= cols)) {
      op = 'T';
      ld = rows == 1 ? cols : sr;
      return true;
    }
    return false;
  };
  char oa, ob, oc;
  int64_t la, lb, lc;
  if (!as_col(g.M, g.N, g.sCm, g.sCn, oc, lc)) return 1;
  if (oc == 'N') {
    if (as_col(g.M, g.K, g.sAm, g.sAk, oa, la) && as_col(g.K, g.N, g.sBk, g.sBn, ob, lb) &&
        itg_libgemm_ok(ctx, ITG_F64, ITG_MODE_NATIVE, oa, ob, g.M, g.N, g.K))
      return itg_libgemm(ctx, oa, ob, g.M, g.N, g.K, g.alpha, (const double*)g.A, la,
                         (const double*)g.B, lb, g.beta, (double*)g.C, lc);
  } else {
    // C^T (n x m, column-major with ld lc) = B^T A^T
    if (as_col(g.N, g.K, g.sBn, g.sBk, ob, lb) && as_col(g.K, g.M, g.sAk, g.sAm, oa, la) &&
        itg_libgemm_ok(ctx, ITG_F64, ITG_MODE_NATIVE, ob, oa, g.N, g.M, g.K))
      return itg_libgemm(ctx, ob, oa, g.N, g.M, g.K, g.alpha, (const double*)g.B, lb,
                         (const double*)g.A, la, g.beta, (double*)g.C, lc);
  }
  return 1;
}

static int scale_output(itg_ctx* ctx, int dtype, int rC, const int64_t* dC, double beta, void* C) {
  int64_t n = 1;
  for (int i = 0; i < rC; ++i) n *= dC[i];
  if (beta == 0.0) return itg_fill(ctx, dtype, n, 0.0, C);
  return itg_scal(ctx, dtype, n, beta, C);
}

extern "C" int itg_contract(itg_ctx* ctx, int dtype, int mode, int rA, const int64_t* dA,
                            const int32_t* lA, const void* A, int rB, const int64_t* dB,
                            const int32_t* lB, const void* B, int rC, const int64_t* dC,
                            const int32_t* lC, void* C, double alpha, double beta) {
  ITG_CHECK_CTX(ctx);
  if (dtype == ITG_C64)
    return itg_c64_contract(ctx, mode, rA, dA, lA, A, rB, dB, lB, B, rC, dC, lC, C, alpha, beta);
  ITG_CHECK_DTYPE(ctx, dtype);
  if (mode < 0 || mode > 2) return itg_fail(ctx, ITG_EARG, "unknown mode %d", mode);
  if (rA < 0 || rB < 0 || rC < 0 || rA > ITG_MAX_RANK || rB > ITG_MAX_RANK || rC > ITG_MAX_RANK)
    return itg_fail(ctx, ITG_EDIM, "rank out of range");
  // validate labels
  auto find = [](const int32_t* l, int r, int32_t x) {
    for (int i = 0; i < r; ++i) if (l[i] == x) return i;
    return -1;
  };
  for (int i = 0; i < rA; ++i) {
    if (find(lA, i, lA[i]) >= 0) return itg_fail(ctx, ITG_EDIM, "repeated label in A");
    if (dA[i] < 0) return itg_fail(ctx, ITG_EDIM, "negative dimension");
    int jb = find(lB, rB, lA[i]), jc = find(lC, rC, lA[i]);
    if (jb >= 0 && jc >= 0)
      return itg_fail(ctx, ITG_EUNSUPPORTED, "label %d in A, B and C (batch modes)", lA[i]);
    if (jb < 0 && jc < 0) return itg_fail(ctx, ITG_EDIM, "label %d of A appears nowhere else", lA[i]);
    if (jb >= 0 && dB[jb] != dA[i]) return itg_fail(ctx, ITG_EDIM, "contracted dims differ for label %d", lA[i]);
    if (jc >= 0 && dC[jc] != dA[i]) return itg_fail(ctx, ITG_EDIM, "dimension mismatch for label %d", lA[i]);
  }
  for (int i = 0; i < rB; ++i) {
    if (find(lB, i, lB[i]) >= 0) return itg_fail(ctx, ITG_EDIM, "repeated label in B");
    if (dB[i] < 0) return itg_fail(ctx, ITG_EDIM, "negative dimension");
    int ja = find(lA, rA, lB[i]), jc = find(lC, rC, lB[i]);
    if (ja < 0 && jc < 0) return itg_fail(ctx, ITG_EDIM, "label %d of B appears nowhere else", lB[i]);
    if (jc >= 0 && dC[jc] != dB[i]) return itg_fail(ctx, ITG_EDIM, "dimension mismatch for label %d", lB[i]);
  }
  for (int i = 0; i < rC; ++i) {
    if (find(lC, i, lC[i]) >= 0) return itg_fail(ctx, ITG_EDIM, "repeated label in C");
    if (find(lA, rA, lC[i]) < 0 && find(lB, rB, lC[i]) < 0)
      return itg_fail(ctx, ITG_EDIM, "output label %d missing from inputs", lC[i]);
  }
  int64_t nC = 1, nK = 1;
  for (int i = 0; i < rC; ++i) nC *= dC[i];
  for (int i = 0; i < rA; ++i) if (find(lB, rB, lA[i]) >= 0) nK *= dA[i];
  if (nC == 0) return ITG_OK;
  if (nK == 0 || alpha == 0.0) return scale_output(ctx, dtype, rC, dC, beta, C);
  // plan lookup: key = ranks, dims and the label pattern
  std::string key;
  key.reserve(16 + 12 * (rA + rB + rC));
  auto app = [&](const void* p, size_t n) { key.append((const char*)p, n); };
  int32_t hdr[3] = {rA, rB, rC};
  app(hdr, sizeof hdr);
  app(dA, rA * sizeof(int64_t)); app(dB, rB * sizeof(int64_t)); app(dC, rC * sizeof(int64_t));
  for (int i = 0; i < rB; ++i) { int32_t x = find(lA, rA, lB[i]); app(&x, 4); }
  for (int i = 0; i < rC; ++i) {
    int32_t x = find(lA, rA, lC[i]);
    if (x < 0) x = 100 + find(lB, rB, lC[i]);
    app(&x, 4);
  }
  itg_plan* p;
  auto it = ctx->plans.find(key);
  if (it != ctx->plans.end()) {
    p = it->second;
  } else {
    int rc = build_plan(ctx, key, rA, dA, lA, rB, dB, lB, rC, dC, lC, &p);
    if (rc) return rc;
  }
  if (p->sic) return launch_sic(ctx, dtype, p, p->swap ? B : A, p->swap ? A : B, C, alpha, beta);
  GettArgs g;
  memset(&g, 0, sizeof g);
  g.A = p->swap ? B : A;
  g.B = p->swap ? A : B;
  g.C = C;
  g.M = p->M; g.N = p->N; g.K = p->K;
  g.sAm = p->sAm; g.sAk = p->sAk; g.sBk = p->sBk; g.sBn = p->sBn; g.sCm = p->sCm; g.sCn = p->sCn;
  auto tp = [&](int64_t o) { return o >= 0 ? p->dtab + o : (const int64_t*)nullptr; };
  g.tAm = tp(p->oAm); g.tAk = tp(p->oAk); g.tBk = tp(p->oBk);
  g.tBn = tp(p->oBn); g.tCm = tp(p->oCm); g.tCn = tp(p->oCn);
  g.alpha = alpha;
  g.beta = beta;
  const bool plain = !g.tAm && !g.tAk && !g.tBk && !g.tBn && !g.tCm && !g.tCn;
  // a tensor with itself over the same modes (a density matrix): half of it
  // is computed
  if (plain && g.A == g.B && g.M == g.N && g.sAm == g.sBn && g.sAk == g.sBk &&
      std::min(g.sCm, g.sCn) == 1 && std::max(g.sCm, g.sCn) >= g.M && mode == ITG_MODE_NATIVE &&
      alpha != 0.0 && beta == 0.0 && g.M >= 256 && band_wins(ctx, mode, g.M)) {
    g.sCm = std::max(g.sCm, g.sCn);
    g.sCn = 1;
    g.band = 1;
    const int rc = launch_gett(ctx, dtype, mode, g, p->akfast, p->bkfast);
    return rc ? rc : mirror_lower(ctx, dtype, g.M, C, g.sCm);
  }
  if (plain && dtype == ITG_F64 && mode == ITG_MODE_NATIVE) {
    int rc = contract_on_lib(ctx, g);
    if (rc != 1) return rc;
  }
  return launch_gett(ctx, dtype, mode, g, p->akfast, p->bkfast);
}

int itg_gemm_internal(itg_ctx* ctx, int dtype, int mode, char ta, char tb, int64_t m, int64_t n,
                      int64_t k, double alpha, const void* A, int64_t lda, const void* B,
                      int64_t ldb, double beta, void* C, int64_t ldc, bool lower_band) {
  if (m == 0 || n == 0) return ITG_OK;
  if (k == 0 || alpha == 0.0) {
    // C = beta*C on an m x n window with leading dimension ldc
    if (ldc == m) {
      if (beta == 0.0) return itg_fill(ctx, dtype, m * n, 0.0, C);
      return itg_scal(ctx, dtype, m * n, beta, C);
    }
    return itg_fail(ctx, ITG_EUNSUPPORTED, "k == 0 with ldc != m");
  }
  bool tA = (ta == 'T' || ta == 't'), tB = (tb == 'T' || tb == 't');
  if (!lower_band && lda >= (tA ? k : m) && ldb >= (tB ? n : k) && ldc >= m &&
      itg_libgemm_ok(ctx, dtype, mode, ta, tb, m, n, k))
    return itg_libgemm(ctx, ta, tb, m, n, k, alpha, (const double*)A, lda, (const double*)B, ldb,
                       beta, (double*)C, ldc);
  GettArgs g;
  memset(&g, 0, sizeof g);
  // C(m,n) at m + n*ldc: its unit stride is m, so compute C^T = B^T A^T
  g.A = B; g.B = A; g.C = C;
  g.M = n; g.N = m; g.K = k;
  // new A = op(B)^T: element (n, k) of op(B)^T = op(B)(k, n)
  g.sAm = tB ? 1 : ldb;  g.sAk = tB ? ldb : 1;
  // new B = op(A)^T: element (k, m) = op(A)(m, k)
  g.sBn = tA ? lda : 1;  g.sBk = tA ? 1 : lda;
  g.sCm = ldc; g.sCn = 1;
  g.alpha = alpha;
  g.beta = beta;
  // the kernel's (tm, tn) is the caller's (column block, row block): the
  // caller's rows >= columns - 1 tile band is tm <= tn + 1
  g.band = (lower_band && m == n) ? 1 : 0;
  bool ak = (g.sAm != 1) && (g.sAk == 1);
  bool bk = (g.sBn != 1) && (g.sBk == 1);
  return launch_gett(ctx, dtype, mode, g, ak, bk);
}

extern "C" int itg_gemm(itg_ctx* ctx, int dtype, int mode, char ta, char tb, int64_t m, int64_t n,
                        int64_t k, double alpha, const void* A, int64_t lda, const void* B,
                        int64_t ldb, double beta, void* C, int64_t ldc) {
  ITG_CHECK_CTX(ctx);
  ITG_CHECK_DTYPE(ctx, dtype);
  if (mode < 0 || mode > 2) return itg_fail(ctx, ITG_EARG, "unknown mode %d", mode);
  if (m < 0 || n < 0 || k < 0 || ldc < std::max<int64_t>(1, m))
    return itg_fail(ctx, ITG_EDIM, "bad GEMM dimensions");
  const bool nt = (ta == 'N' || ta == 'n') && (tb == 'T' || tb == 't');
  const bool tn = (ta == 'T' || ta == 't') && (tb == 'N' || tb == 'n');
  if (A == B && lda == ldb && m == n && m >= 256 && k > 0 && beta == 0.0 && alpha != 0.0 &&
      (nt || tn)) {
    // C = alpha A A^T (or A^T A), the density matrix of a bond, exactly symmetric
    const int rc = itg_gemm_internal(ctx, dtype, mode, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta,
                                     C, ldc, band_wins(ctx, mode, m));
    return rc ? rc : mirror_lower(ctx, dtype, m, C, ldc);
  }
  return itg_gemm_internal(ctx, dtype, mode, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

int itg_gett_launch(itg_ctx* ctx, int dtype, int mode, GettArgs* g, bool ak, bool bk) {
  if (g->M <= 0 || g->N <= 0) return ITG_OK;
  return launch_gett(ctx, dtype, mode, *g, ak, bk);
}
