// LDS layout of the Heff W pass (heff.hip), shared with a CPU test: X as rows
// of one q each, the outputs o along a row, 16-wide column tiles taken NT at a
// time.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define ITG_HD __host__ __device__
#else
#define ITG_HD
#endif

// doubles per row: whole column tiles, an odd number of them, so that the four
// rows a product reads start half the banks apart
ITG_HD static inline int wpass_ldo(int O) {
  const int ot = (O + 15) / 16;
  return (ot % 2 == 0 ? ot + 1 : ot) * 16;
}

ITG_HD static inline int wpass_rows(int Q) { return (Q + 3) / 4 * 4; }

// where the products of column tile o0 + j find X(q, 16 (o0 + j) + lr)
ITG_HD static inline int wpass_at(int q, int ldo, int o0, int j, int lr) {
  return q * ldo + 16 * (o0 + j) + lr;
}

// doubles in all: the last NT tiles of a row reach past it when the tiles are
// no multiple of NT, into the next row or, from the last one, these
ITG_HD static inline int wpass_doubles(int Q, int O, int nt) {
  return wpass_rows(Q) * wpass_ldo(O) + 16 * (nt - 1);
}

// column tiles a wave takes at a time
ITG_HD static inline int wpass_nt(int64_t O) {
  return O <= 16 ? 1 : O <= 32 ? 2 : 4;
}

constexpr int64_t WPASS_LDS = 65536;   // bytes of X per launch

// operators the apply takes (w = 14, d = 2: 56 (64 + 56) = 6720); Q <= 126, so
// that X has room for at least 16 outputs
ITG_HD static inline bool wpass_takes(int64_t Q, int64_t O) { return Q * (64 + O) <= 8192; }

// outputs per launch: as many as X has room for (all of them but for an MPO of
// thousands of channels and d = 1)
ITG_HD static inline int wpass_outputs(int Q, int O, int nt) {
  int os = O;
  while (os > 16 && wpass_doubles(Q, os, nt) * (int64_t)sizeof(double) > WPASS_LDS)
    os = (os / 2 + 15) / 16 * 16;
  return os;
}
