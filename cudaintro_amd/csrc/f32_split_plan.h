// Launch planning of the fp32 tiles on the bf16 matrix instructions (f32_split_tile.h), as plain host
// functions of sizes.
#pragma once
#include "any_plan.h"

namespace cig {
namespace split32 {

struct Plan {
  int rows;          // of a tile: 64, 96 or 128; 0: no plan
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
// units at work (the chip's power limit); a round: ramp and epilogue; the operands by the MB, the
// reduction behind K ranges.  Fitted to 35092 timed plans of 10198 sizes (M 16..20000, N 16..16384, K
// 17..16384, log-uniform, up to 1.4e11 operations): rms error 4 %; the plan it likes best is 0.2 %
// slower than the best one timed, on average.
struct Cost {
  double stage, stage_chip, round;
};
constexpr Cost COST[3] = {{0.554, 0.379, 5.25}, {0.670, 0.523, 6.32}, {0.807, 0.648, 7.51}};
constexpr double START_US = 2.47, IN_MB = 0.0174, REDUCE_US = 1.26, REDUCE_MB = 0.153;
constexpr Cost cost_of(int rows) { return COST[rows / 32 - 2]; }

inline double launch_us(int64_t M, int64_t N, int64_t K, int cus, int rows, int ranges) {
  const Cost c = cost_of(rows);
  int64_t range_k = 0;
  const int sp = k_ranges(K, ranges, &range_k);
  const int64_t tiles = any::div_up(M, rows) * any::div_up(N, tile::BN) * sp;
  const double stages = (double)range_k / 16 + 1, mn = (double)M * (double)N * 4e-6;
  double us = START_US + (double)(tiles / cus) * (stages * (c.stage + c.stage_chip) + c.round);
  if (tiles % cus) us += stages * (c.stage + c.stage_chip * (double)(tiles % cus) / cus) + c.round;
  us += IN_MB * (double)(M + N) * (double)K * 4e-6;
  if (sp > 1) us += REDUCE_US + REDUCE_MB * mn * (sp + 1);
  return us;
}

// The longest sum of k that a result may be made of, where the other kernel adds up `sum_length`.  Of equally long
// sums the error here is at most 0.71 times the fp32 instructions' (0.83 and 1.00 where two products or one
// make the result, whose errors do not grow); that of positive operands grows with the length (over K in one
// sum, against the fp32 instructions over six ranges of it: 1.7 to 4.3 times).  (Where the other kernel takes two
// launches, its length is the first one's, which has most of the columns.)
constexpr int64_t range_limit(int64_t sum_length) { return sum_length + sum_length / 4; }

// No single launch over these sizes takes less: the stages of all tiles spread evenly over the units, on the height
// that needs least for a row, and the terms that no plan avoids.
inline double least_us(int64_t M, int64_t N, int64_t K, int cus, int rows) {
  const Cost c = cost_of(rows);
  const double tiles = (double)(any::div_up(M, rows) * any::div_up(N, tile::BN));
  return START_US + tiles * ((double)K / 16) / cus * (c.stage + c.stage_chip) + c.round +
         IN_MB * (double)(M + N) * (double)K * 4e-6;
}

// The best single launch below `*est`, which it lowers; `sum_length`: of the kernel this one takes the place of.
// What cannot be below it is not looked at: planning is host time (4000 random calls, M 1..8192, N and K 16..16384,
// all of the choice: 0.31 us on average and 3.1 for one in a hundred with every plan, 0.16 and 1.6 now, most of it the
// other kernels' estimates).
inline Plan best_launch(int64_t M, int64_t N, int64_t K, int64_t sum_length, int cus, size_t partial_bytes,
                        double* est) {
  Plan best{0, 1, 0, 0};
  const int64_t limit = range_limit(sum_length);
  const int fewest = (int)any::at_most((double)any::div_up(K, limit > 0 ? limit : 1), 33);
  for (int rows = 64; rows <= 128; rows += 32) {
    if (rows > 64 && rows - 32 >= M) break;  // a lower height already covers M
    const int64_t tiles = any::div_up(M, rows) * any::div_up(N, tile::BN);
    const double least = least_us(M, N, K, cus, rows), mn = (double)M * (double)N * 4e-6;
    int last = 0;
    for (int wanted = fewest > 1 ? fewest : 1; wanted <= 32; ++wanted) {
      if (least + (wanted > 1 ? REDUCE_US + REDUCE_MB * mn * (last + 1) : 0.0) >= *est) break;
      int64_t range_k = 0;
      const int sp = k_ranges(K, wanted, &range_k);
      if (sp > 1 && (tiles * sp > 2 * (int64_t)cus || range_k < 64 ||
                     (size_t)sp * (size_t)M * (size_t)(any::div_up(N, 32) * 32) * 4 > partial_bytes))
        break;
      if (sp == last) continue;
      last = sp;
      if (range_k > limit) continue;
      const double us = launch_us(M, N, K, cus, rows, sp);
      if (us < *est) *est = us, best = Plan{rows, sp, 0, 0};
    }
  }
  return best;
}

// That, or the columns that fill whole rounds on one height and the others by themselves; `*est` as there.
inline Plan best(int64_t M, int64_t N, int64_t K, int64_t sum_length, int cus, size_t partial_bytes,
                 double* est) {
  Plan b = best_launch(M, N, K, sum_length, cus, partial_bytes, est);
  const int64_t tiles_n = any::div_up(N, tile::BN);
  for (int rows = 96; rows <= 128; rows += 32) {
    const int64_t tiles_m = any::div_up(M, rows);
    if (tiles_m > cus || K > range_limit(sum_length)) continue;
    const int64_t per_round = cus / tiles_m, cols = tiles_n / per_round * per_round;
    if (cols <= 0 || cols >= tiles_n) continue;
    const double first = launch_us(M, cols * tile::BN, K, cus, rows, 1);
    if (first >= *est) continue;
    double us = *est - first;
    const Plan rest = best_launch(M, N - cols * tile::BN, K, sum_length, cus, partial_bytes, &us);
    if (rest.rows) *est = first + us, b = Plan{rest.rows, rest.ranges, cols * tile::BN, rows};
  }
  return b;
}

}  // namespace split32
}  // namespace cig
