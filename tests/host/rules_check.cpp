// The library's launch rules (csrc/rules.h) behind a C interface, for the tests
// that name the kernel they are written for.
#include "rules.h"

extern "C" {

int rule_mxg_wide(int members, int tiles_m, int N, int mats, int fp4, int kpad) {
  return wv::mxg_wide(members, tiles_m, N, mats, fp4 != 0, kpad) ? 1 : 0;
}

int rule_mxg_weights_fit(long long N, long long pitch) {
  return wv::mxg_weights_fit(N, pitch) ? 1 : 0;
}

// kernel, waves, sub-blocks ahead, gemm tile (tm, tn), gemm rows of one run
void rule_format_plan(int fmt, int rows, int nsub, int batch, long long ws_bytes, long long* out) {
  const wv::FmtPlan p = wv::format_plan(fmt, rows, nsub, batch);
  const wv::FmtTile t = wv::format_tile(rows, batch);
  out[0] = (int)p.kernel, out[1] = p.waves, out[2] = p.depth, out[3] = t.tm, out[4] = t.tn;
  out[5] = wv::format_run_rows(fmt, nsub, (size_t)ws_bytes);
}

}  // extern "C"
