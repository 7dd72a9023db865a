// Rules that choose a launch shape from sizes alone: plain C++, shared by the
// kernels' host code, the layers and the host tests.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace wv {

constexpr long kCus = 256;

// Wide tiles of the large-tile product (128 activation rows x 256 staged weight
// rows per step, 128 per matrix of two) move half the activation bytes per
// MFMA of the narrow ones (128). Taken when they still give every CU a workgroup
// and N is a multiple of their width (the weight rows and scales are padded to
// 128), but not where they leave the second of two rounds over the CUs half empty
// or worse: 257 to 384 wide tiles are two rounds, twice as many narrow ones
// three. A wide tile takes 1.6 times a narrow one's time, of FP4 weights (whose
// wide loop has fewer bytes to wait for) 1.4 beyond 1536 columns; there two wide
// rounds are the shorter ones. us, wide / narrow: 4096 rows x 1024 x 3072 E4M3 52.1 /
// 46.8, FP4 41.7 / 38.3; x 4096 x 3072 E4M3 165 / 155, FP4 130 / 140.
inline bool mxg_wide(int members, int tiles_m, int N, int mats, bool fp4, int kpad) {
  const int bn = 256 / mats;
  const long tiles = (long)members * tiles_m * (N / bn);
  if (N % bn != 0 || tiles < kCus) return false;
  const bool half_empty = tiles > kCus && 2 * tiles <= 3 * kCus;
  return !half_empty || (fp4 && kpad > 1536);
}

// The large-tile product addresses its weight codes with 32-bit offsets: N rows
// (padded to a wide tile) of `pitch` bytes stay below 2 GiB.
inline bool mxg_weights_fit(int64_t N, int64_t pitch) {
  return (N + 255) / 256 * 256 * pitch < (1ll << 31);
}

}  // namespace wv
