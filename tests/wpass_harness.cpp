// The W pass's reads of X in LDS (itensorsgpu.jl_amd/csrc/wpass_core.h), walked
// on the CPU in the kernel's loops. Test infrastructure only.
#include "wpass_core.h"

// largest index read by a launch of O outputs, nt column tiles at a time
extern "C" int64_t wpass_last_read(int Q, int O, int nt) {
  int64_t last = -1;
  const int ldo = wpass_ldo(O), ot = (O + 15) / 16, kt = (Q + 3) / 4;
  for (int o0 = 0; o0 < ot; o0 += nt)
    for (int k = 0; k < kt; ++k)
      for (int lg = 0; lg < 4; ++lg)
        for (int j = 0; j < nt; ++j) {
          const int64_t x = wpass_at(4 * k + lg, ldo, o0, j, 15);
          if (x > last) last = x;
        }
  return last;
}

extern "C" int64_t wpass_size(int Q, int O, int nt) { return wpass_doubles(Q, O, nt); }
extern "C" int wpass_tiles(int64_t O) { return wpass_nt(O); }
extern "C" int wpass_slice(int Q, int O, int nt) { return wpass_outputs(Q, O, nt); }
extern "C" int wpass_taken(int64_t Q, int64_t O) { return wpass_takes(Q, O) ? 1 : 0; }
