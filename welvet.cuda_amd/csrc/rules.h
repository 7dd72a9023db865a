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

// ---- packed block formats ----
// QuantFormat ids: the reference's enum (include/welvet/weights.hpp:12-15)
// holds only None; the other values follow the order of its format table
// (README.md:361-383).
enum QuantFormat : int32_t {
  kFmtNone = 0, kQ8_0 = 1, kQ4_0 = 2, kQ4_1 = 3, kQ5_0 = 4, kQ5_1 = 5, kQ2_K = 6, kQ3_K = 7,
  kQ4_K = 8, kQ5_K = 9, kQ6_K = 10, kIQ4_NL = 16, kIQ4_XS = 17, kFmtLast = 20
};

// y = d (c x) + off (sum x): the formats with an offset per sub-block
constexpr bool fmt_affine(int fmt) {
  return fmt == kQ4_1 || fmt == kQ5_1 || fmt == kQ2_K || fmt == kQ4_K || fmt == kQ5_K;
}

// operand bytes of 32 batch rows x 32 elements in the matrix-core product's scratch
constexpr int fmt_split_bytes(bool affine) { return affine ? 7168 : 6144; }
constexpr size_t kFmtWsBytes = 64ull << 20;
inline size_t format_ws_bytes(int nsub, int batch) {
  if (batch <= 16) return 0;
  const size_t n = (size_t)((batch + 31) / 32) * nsub * fmt_split_bytes(true);
  return n < kFmtWsBytes ? n : kFmtWsBytes;
}

// Batch rows from which the matrix cores take the product. 4096 x 4096 at 4 and
// 6 rows, us, the per-row kernel against the matrix cores: Q8_0 16.3 / 10.0 and
// 21.7 / 10.4, Q4_0 11.6 / 9.8 and 13.8 / 10.1, Q4_1 10.1 / 11.6 and 13.8 /
// 11.9, Q2_K 11.5 / 13.6 and 14.3 / 14.0 (the others like Q4_0).
constexpr int format_rows_batch(int fmt) {
  return fmt == kQ2_K ? 6 : fmt == kQ4_1 || fmt == kQ5_1 ? 5 : 4;
}

// The kernel of a product of `batch` rows with a matrix of `rows` x 32 nsub.
enum class FmtKernel : int { kPerRow = 0, kRows = 1, kGemm = 2 };
struct FmtPlan {
  FmtKernel kernel;
  int waves, depth;  // kRows: waves per workgroup, sub-blocks a wave loads ahead
};

inline FmtPlan format_plan(int fmt, int rows, int nsub, int batch) {
  FmtPlan p = {FmtKernel::kPerRow, 0, 0};
  // The per-row kernel's time goes with the rows times batch rows times chunks of
  // 64 sub-blocks (partly filled ones count whole), the matrix-core kernel's
  // with the sub-blocks that one workgroup walks. us, per-row / matrix cores
  // (Q4_0 and Q6_K): 768 x 448 at 6 rows 3.7 / 4.1 and 3.9 / 4.6, 2048 x 2048 at 4
  // rows 4.9 / 5.5 and 5.4 / 6.7, 768 x 6400 at 4 rows 7.7 / 5.5 and 11.1 / 6.6,
  // 8192 x 256 at 6 rows 4.8 / 14.6 and 5.3 / 19.4. Only below 8 rows: from there
  // an infinity of x meets each dequantized weight (fmt_store), where the
  // per-row kernel's offset sums make it NaN.
  const int chunks = (nsub + 63) / 64;
  const int64_t per_row = (int64_t)rows * batch * chunks;
  const bool small = batch < 8 && per_row <= (nsub > 40 ? 200 * (int64_t)nsub : 8192);
  if (small || batch < format_rows_batch(fmt)) return p;
  // Above 16 batch rows the split and the larger tiles are two launches (6.8 us
  // at the least): one as long as every workgroup of 16 x 16 has a CU to itself,
  // or they have no more to do than that many of 2432 columns, a workgroup's
  // start and end counted as 4 sub-blocks. us, one launch / two, Q4_0 and Q6_K: 512 x 256
  // at 300 rows (304 workgroups) 4.5 / 7.7 and 5.0 / 8.1, at 1000 rows (1008) 6.7 /
  // 11.6 and 7.5 / 11.8, 1024 x 1024 at 100 rows (448) 6.8 / 8.4 and 7.5 / 9.0, at 300
  // rows (1216) 13.0 / 12.0 and 14.9 / 13.3, 768 x 4096 at 100 rows (1792) 13.3 / 9.6
  // and 16.1 / 11.0, 256 x 8192 at 64 rows (2048) Q6_K 8.4 / 8.0.
  const int64_t blocks = ((int64_t)rows + 15) / 16 * ((batch + 15) / 16);
  if (batch <= 16 || blocks <= kCus || blocks * (nsub + 4) <= 80 * kCus) {
    p.kernel = FmtKernel::kRows;
    // Waves by the sub-blocks they split, 8 rows of Q4_0, us with 4 / 8 / 16 waves:
    // 512 x 256 4.1 / 4.1 / 5.4 (Q4_K 3.9 / 4.7 / 6.6), 1024 x 1024 4.5 / 4.1 /
    // 5.5, 768 x 6400 6.0 / 5.7 / 9.2, 2048 x 2048 6.8 / 5.8 / 5.6, 2048 x 4096 6.8 /
    // 5.9 / 5.7. A wave loads all of its sub-blocks ahead, or equal runs of at most
    // 4: what a run holds past the last one is loaded for nothing (256 x 8192 at 16
    // rows, 2 sub-blocks a wave, with runs of 4 / 2: Q4_0 4.6 / 3.6, Q6_K 5.2 / 3.8;
    // 768 x 448, 3 a wave, with 4 / 3: Q6_K 4.9 / 4.3, Q2_K 5.1 / 4.4).
    // Where each workgroup has a CU to itself 16 waves from 32 sub-blocks on, 40 for
    // the formats that decode in fewer steps (1024 x 1024 at 8 rows, 8 / 16 waves:
    // Q4_K 4.8 / 4.5, Q8_0 3.8 / 3.8; 1280 x 300 Q6_K 5.9 / 5.4, Q4_1 5.5 / 5.2).
    const int most8 = blocks > kCus ? 64 : fmt <= kQ5_1 ? 40 : 32;
    p.waves = nsub <= 16 ? 4 : nsub < most8 ? 8 : 16;
    const int per = (nsub + p.waves - 1) / p.waves, runs = (per + 3) / 4;
    p.depth = (per + runs - 1) / runs;
    if (p.depth < 2) p.depth = 2;
    return p;
  }
  p.kernel = FmtKernel::kGemm;
  return p;
}

// The gemm's tile, in units of 32 batch rows x 32 weight rows.
struct FmtTile {
  int tm, tn;
};

// The largest tile (a decoded weight and a loaded term feed more products)
// that still reaches three quarters of the 256 CUs. 4096 x 4096 Q4_0, us at
// tiles 1 x 1 / 1 x 2 / 2 x 2 / 2 x 4: 64 rows 15.9 / 19.0 / 31.9 / 49.0, 128
// rows 26.6 / 22.1 / 34.1 / 49.3, 256 rows 50.4 / 39.7 / 40.1 / 52.5, 512 rows
// 114 / 75 / 74 / 62.
inline FmtTile format_tile(int rows, int batch) {
  const auto fills = [&](int tm, int tn) {
    return (int64_t)((batch + 32 * tm - 1) / (32 * tm)) * ((rows + 32 * tn - 1) / (32 * tn)) >= 192;
  };
  if (fills(2, 4)) return {2, 4};
  if (fills(2, 2)) return {2, 2};
  if (fills(1, 2)) return {1, 2};
  return {1, 1};
}

// Batch rows of one run of the gemm: as many as the scratch holds terms of.
inline int64_t format_run_rows(int fmt, int nsub, size_t ws_bytes) {
  return (int64_t)(ws_bytes / ((size_t)nsub * fmt_split_bytes(fmt_affine(fmt)))) * 32;
}

}  // namespace wv
