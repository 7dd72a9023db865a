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

}  // extern "C"
