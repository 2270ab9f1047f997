// Launch planning of the fp32 tiles on the bf16 matrix instructions (f32_split_tile.h), as plain host
// functions of sizes.
#pragma once
#include "any_plan.h"

namespace cig {
namespace split32 {

struct Plan {
  int rows;          // of a tile: 64, 96 .. 256; 0: no plan
  int ranges;        // of K
  int64_t first_cols;  // > 0: these columns first, unsplit, on tiles of first_rows; the others by the above
  int first_rows;
};

// K ranges of whole stages (16 of k), the last with what is left; every one of at least 17, what the
// kernel takes.
inline int k_ranges(int64_t K, int wanted, int64_t* range_k) {
  for (int64_t n = wanted; n > 1; --n) {
    const int64_t rk = (any::div_up(K, n) + 15) / 16 * 16;
    const int64_t ranges = any::div_up(K, rk);
    if (rk >= 32 && ranges > 1 && K - (ranges - 1) * rk >= 17) {
      *range_k = rk;
      return (int)ranges;
    }
  }
  *range_k = K;
  return 1;
}

// Sizes the kernel can run: a whole stage beside the 1..16 of k it takes one by one, columns in pairs, lane
// offsets of 32 bits.
inline bool ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb) {
  return M >= 1 && N >= 2 && K >= 17 && M <= 2147483647LL - 255 && N <= 2147483647LL - 255 &&
         K <= 2147483647LL && any::div_up(M, 64) * any::div_up(N, 256) <= 2147483647LL &&
         lda * 4 * 256 < (1LL << 31) && ldb * 4 * 256 < (1LL << 31);
}

// us of one launch.  A stage of a round of workgroups: a part of its own and a part that grows with the
// units at work (the chip's power limit); a round: ramp and epilogue; the output and the operands by
// the MB, the reduction behind K ranges.  Fitted to 6600 timed plans of 1000 sizes (M 16..20000, N 16..
// 16384, K 17..16384, log-uniform, up to 1.4e11 operations): rms error 5 %; the plan it likes best is 0.5 %
// slower than the best one timed, on average.
struct Cost {
  double stage, stage_chip, round;
};
constexpr Cost COST[7] = {{0.647, 0.131, 4.52}, {0.696, 0.225, 5.38}, {0.852, 0.274, 6.44}, {1.038, 0.386, 6.59},
                          {1.117, 0.467, 7.72}, {1.292, 0.499, 8.22}, {1.419, 0.561, 9.36}};
constexpr double START_US = 2.54, OUT_MB = 0.0523, IN_MB = 0.0141, REDUCE_US = 2.65, REDUCE_MB = 0.155;
constexpr Cost cost_of(int rows) { return COST[rows / 32 - 2]; }

inline double launch_us(int64_t M, int64_t N, int64_t K, int cus, int rows, int ranges) {
  const Cost c = cost_of(rows);
  int64_t range_k = 0;
  const int sp = k_ranges(K, ranges, &range_k);
  const int64_t tiles = any::div_up(M, rows) * any::div_up(N, tile::BN) * sp;
  const double stages = (double)range_k / 16 + 1, mn = (double)M * (double)N * 4e-6;
  double us = START_US + (double)(tiles / cus) * (stages * (c.stage + c.stage_chip) + c.round);
  if (tiles % cus) us += stages * (c.stage + c.stage_chip * (double)(tiles % cus) / cus) + c.round;
  us += OUT_MB * mn * sp + IN_MB * (double)(M + N) * (double)K * 4e-6;
  if (sp > 1) us += REDUCE_US + REDUCE_MB * mn * (sp + 1);
  return us;
}

// The longest sum of k that a result may be made of, as the fp32 instructions add it up, where the tiles
// of this height are to round no more: with one running sum of a block (above 128 rows) their error is 0.75
// to 0.93 of the fp32 instructions', with two 0.32 to 0.4, and it grows with the square root of the length.
constexpr int64_t range_limit(int rows, int64_t sum_length) { return rows > 128 ? sum_length : 6 * sum_length; }

// The best single launch; `sum_length`: of the kernel this one takes the place of.
inline Plan best_launch(int64_t M, int64_t N, int64_t K, int64_t sum_length, int cus, size_t partial_bytes,
                        double* est) {
  Plan best{0, 1, 0, 0};
  *est = 1e30;
  for (int rows = 64; rows <= 256; rows += 32) {
    if (rows > 64 && rows - 32 >= M) break;  // a lower height already covers M
    const int64_t tiles = any::div_up(M, rows) * any::div_up(N, tile::BN);
    int last = 0;
    for (int wanted = 1; wanted <= 32; ++wanted) {
      int64_t range_k = 0;
      const int sp = k_ranges(K, wanted, &range_k);
      if (sp > 1 && (tiles * sp > 2 * (int64_t)cus || range_k < 64 ||
                     (size_t)sp * (size_t)M * (size_t)(any::div_up(N, 32) * 32) * 4 > partial_bytes))
        break;
      if (sp == last) continue;
      last = sp;
      if (range_k > range_limit(rows, sum_length)) continue;
      const double us = launch_us(M, N, K, cus, rows, sp);
      if (us < *est) *est = us, best = Plan{rows, sp, 0, 0};
    }
  }
  return best;
}

// That, or the columns that fill whole rounds on one height and the others by themselves.
inline Plan best(int64_t M, int64_t N, int64_t K, int64_t sum_length, int cus, size_t partial_bytes,
                 double* est) {
  Plan b = best_launch(M, N, K, sum_length, cus, partial_bytes, est);
  const int64_t tiles_n = any::div_up(N, tile::BN);
  for (int rows = 96; rows <= 256; rows += 32) {
    const int64_t tiles_m = any::div_up(M, rows);
    if (tiles_m > cus || K > range_limit(rows, sum_length)) continue;
    const int64_t per_round = cus / tiles_m, cols = tiles_n / per_round * per_round;
    if (cols <= 0 || cols >= tiles_n) continue;
    const double first = launch_us(M, cols * tile::BN, K, cus, rows, 1);
    if (first >= *est) continue;
    double us = 0;
    const Plan rest = best_launch(M, N - cols * tile::BN, K, sum_length, cus, partial_bytes, &us);
    if (rest.rows && first + us < *est) *est = first + us, b = Plan{rest.rows, rest.ranges, cols * tile::BN, rows};
  }
  return b;
}

}  // namespace split32
}  // namespace cig
