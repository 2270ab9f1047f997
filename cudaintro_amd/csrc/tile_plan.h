// Launch planning of the LDS-DMA tile kernel (mfma_tile.h), as plain host functions of sizes
// so that a host-only test can check them: the K ranges of a split launch, the estimate that
// ranks (tile height, K ranges) plans, and the tile height of plans of several rounds.
#pragma once
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace cig {
namespace tile {

constexpr int BM = 256, BN = 256;          // the largest output tile
constexpr int KB = 64;                     // bytes of k per stage, per row

// Whether the epilogue of the tile kernel stores C with streaming stores: where a row of C is made of
// whole 16-byte pieces, but for fp32's waves of 64 columns (nt = 2) only where it begins with a line.
// `first_row`, `row_step`: C's address and bytes per row; any: the any-alignment form (the other one's
// rows are whole pieces); rows: of the tile.  Such a wave stores 256 bytes of a row at a time; if the
// row does not begin with a line, both ends are half lines whose other half is another wave's, and
// streaming stores do not wait for it in the L2.  us, streaming -> plain: 4096 x 4100 x 64 49.5 -> 38.1
// (waves of 128 columns 44.0), 8192 x 6532 x 64 126.8 -> 107.7 (115.7), x 256 260.5 -> 239 (248.4); 75
// sizes whose rows are whole pieces (M 100..20000, K 64..1024) 1.08 times as fast together, one 3 %
// slower.  Rows of whole lines: plain ones up to 6 % slower.  64-row tiles, too: 20 sizes 0.99 times.
constexpr bool store_streams(int64_t first_row, int64_t row_step, bool any, int nt, int rows) {
  return nt == 2 && rows > 64 ? ((first_row | row_step) & 127) == 0
                              : !any || ((first_row | row_step) & 15) == 0;
}

// K ranges of a split-K launch: `wanted` ranges over K_bytes of k become ranges of an even
// number of whole stages (operand rows are fetched as 128-byte lines, two stages: an odd range
// would start every later one in the middle of a line), the last one holding what is left.
// Returns the number of ranges that gives (<= wanted) and the stages of each but the last.
inline int k_ranges(int64_t K_bytes, int wanted, int64_t* range_stages) {
  const int64_t kts = (K_bytes + KB - 1) / KB;
  if (wanted <= 1 || kts < 2) {
    *range_stages = kts;
    return 1;
  }
  int64_t rs = (kts + wanted - 1) / wanted;
  rs += rs & 1;
  *range_stages = rs;
  return (int)((kts + rs - 1) / rs);
}

// Plan for a problem that fits one round of 256-row tiles: tile height and number of K
// ranges, by estimated time.  The estimate has the terms that decide between such plans; its
// constants were chosen so that it ranks the plans of a timed sweep well (759 problems: batch
// sizes 33..2048 over weight shapes of common decoder layers, bf16, int8 in both layouts and
// fp32, every tile height x 1..32 ranges timed; tests/test_tile_plan.py checks the ranking
// against those timings) and, second, so that it stays near the times themselves (rms error 12 %
// on plans within 30 % of the best).  The plan it picks is 2 % slower than the best plan timed
// on average, on those problems and on 237 others first timed afterwards.
//   One round of workgroups = a fixed cost + stages per range x cost of a stage + this round's
//   share of the memory traffic (both operands once, plus the partial sums or the output,
//   weighted) at a streaming rate; a last, partly filled round is priced by its own number of
//   workgroups.
//   A split plan adds the reduction launch as measured: max(4.75, 1.1 + bytes / 5.3 TB/s) us
//   for `splits` fp32 partial matrices read and one output written.
// A stage costs a workgroup a part that does not depend on the tile height (it waits for its
// operands: with three stages in flight the wait per stage is a third of the memory latency,
// less when B sits in the L2 / Infinity Cache) plus a part per 64 rows (LDS reads and matrix
// instructions; fp32, whose matrix instructions are 16 times slower, is the one layout where
// that part dominates).
struct SmallPlan {
  int mt;
  int splits;
};
struct StageCost {
  double fixed_us;     // per 64-byte stage, whatever the tile height (B streams from HBM)
  double per_64_rows_us;
};
// by operand layout: 16-bit K x N, int8 N x K, int8 K x N, fp32 K x N
constexpr StageCost STAGE_COST_KN16{0.234, 0.032};
constexpr StageCost STAGE_COST_NK8{0.327, 0.008};
constexpr StageCost STAGE_COST_KN8{0.261, 0.037};
constexpr StageCost STAGE_COST_KN32{0.061, 0.746};
struct PlanCost {
  // (the fixed cost of a round came out near zero: what a launch costs whatever the plan does
  // not help to choose one)
  static constexpr double ROUND_US = 0.05;         // ramp and epilogue of a round of workgroups
  static constexpr double LATER_ROUND_US = 0.05;   // the same for a partly filled last round
  static constexpr double HBM_TB_S = 9.0;
  static constexpr double PARTIAL_WEIGHT = 3.43;   // bytes of partial sums / output, weighted
  static constexpr double RESIDENT_FIXED = 0.857;  // factor on StageCost::fixed_us, B <= 16 MiB
  static constexpr int MIN_RANGE_STAGES = 8;
  static constexpr int MAX_ROUNDS_SPLIT = 3;
};
// The estimate for tiles of `rows` rows.
inline double plan_us_rows(int64_t M, int64_t N, int64_t K_bytes, int out_bytes, StageCost sc,
                           bool streamed, int cus, int rows, int sp, int64_t range_stages) {
  const int64_t tiles = ((M + rows - 1) / rows) * ((N + BN - 1) / BN);
  const int64_t wgs = tiles * sp, full = wgs / cus, rem = wgs % cus;
  const double stage =
      (streamed ? sc.fixed_us : sc.fixed_us * PlanCost::RESIDENT_FIXED) + sc.per_64_rows_us * rows / 64;
  const double mn = (double)M * (double)N;
  const double hbm_bytes = (double)(N + M) * (double)K_bytes +
                           PlanCost::PARTIAL_WEIGHT * (sp > 1 ? sp * mn * 4.0 : mn * out_bytes);
  auto round_body = [&](int64_t active) {
    return stage * (double)range_stages +
           hbm_bytes * (double)active / (double)wgs / (PlanCost::HBM_TB_S * 1e6);
  };
  double us;
  if (full > 0) {
    us = (double)full * (PlanCost::ROUND_US + round_body(cus));
    if (rem > 0) us += PlanCost::LATER_ROUND_US + round_body(rem);
  } else {
    us = PlanCost::ROUND_US + round_body(rem);
  }
  if (sp > 1) {
    const double reduce = 1.1 + (sp * 4.0 + out_bytes) * mn / 5.3e6;
    us += reduce > 4.75 ? reduce : 4.75;
  }
  return us;
}

inline double plan_us(int64_t M, int64_t N, int64_t K_bytes, int out_bytes, StageCost sc,
                      bool streamed, int cus, int mt, int sp, int64_t range_stages) {
  return plan_us_rows(M, N, K_bytes, out_bytes, sc, streamed, cus, 64 * mt, sp, range_stages);
}

// `partial_bytes` = room for partial sums (0: no split plans).  `est_us`, if given, receives the
// estimate of the plan returned.
inline SmallPlan plan_small(int cus, size_t partial_bytes, int64_t M, int64_t N, int64_t K_bytes,
                            int out_bytes, StageCost sc, int64_t b_bytes,
                            double* est_us = nullptr) {
  const bool streamed = b_bytes > (16LL << 20);
  if (cus <= 0) cus = 256;
  SmallPlan best{0, 1};
  double best_us = 1e30;
  for (int mt : {4, 3, 2, 1}) {
    if (mt > 1 && 64 * (mt - 1) >= M) continue;  // the next lower height already covers M
    const int64_t tiles = ((M + 64 * mt - 1) / (64 * mt)) * ((N + BN - 1) / BN);
    int last_sp = 0;
    for (int wanted = 1; wanted <= 32; ++wanted) {
      int64_t range_stages = 0;
      const int sp = k_ranges(K_bytes, wanted, &range_stages);
      if (sp == last_sp) continue;
      last_sp = sp;
      if (sp > 1) {
        if (range_stages < PlanCost::MIN_RANGE_STAGES) break;
        if (tiles * sp > (int64_t)PlanCost::MAX_ROUNDS_SPLIT * cus) break;
        if ((size_t)sp * (size_t)M * (size_t)N * 4 > partial_bytes) break;
      }
      const double us = plan_us(M, N, K_bytes, out_bytes, sc, streamed, cus, mt, sp, range_stages);
      if (us < best_us) {
        best_us = us;
        best = SmallPlan{mt, sp};
      }
    }
  }
  if (est_us) *est_us = best_us;
  return best;
}

// fp32, whose tiles may have any multiple of 32 rows: the height for `plan`'s number of K ranges that
// the same estimate likes best, among the plan's own and all that lie between the multiples of 64.
// (83 x 6752 x 4352: 96 rows in place of 128.)  `est_us`, if given, receives that height's estimate.
inline int plan_small_rows32(int cus, int64_t M, int64_t N, int64_t K_bytes,
                             int out_bytes, StageCost sc, int64_t b_bytes, SmallPlan plan,
                             double* est_us = nullptr) {
  const bool streamed = b_bytes > (16LL << 20);
  if (cus <= 0) cus = 256;
  int64_t range_stages = 0;
  const int sp = k_ranges(K_bytes, plan.splits, &range_stages);
  int best = 64 * plan.mt;
  double best_us = plan_us_rows(M, N, K_bytes, out_bytes, sc, streamed, cus, best, sp, range_stages);
  for (int rows : {96, 160, 224}) {
    if (rows - 32 >= M) break;  // a lower height already covers M
    const double us =
        plan_us_rows(M, N, K_bytes, out_bytes, sc, streamed, cus, rows, sp, range_stages);
    if (us < best_us) best_us = us, best = rows;
  }
  if (est_us) *est_us = best_us;
  return best;
}

// Cost of one tile of 64*mt rows in a plan of several rounds (compute bound), in units of a
// quarter of the 256-row tile's: a fixed part (the B panel is fetched whatever the height) plus
// a part per 64 rows.  One round of 256 tiles, N = 4096, K = 1024..4096, 16-bit and int8:
// 4.0 / 3.1-3.2 / 2.3 / 1.6-1.8.  fp32, whose matrix instructions are 16 times slower, pays
// almost by the row (TILE_UNITS_F32): 5120 x 4096 x 4096 on 64-row tiles 1179 us against 1362 on
// 192-row ones, 7000 x 4096 x 11008 4481 against 4875 on 256-row ones, 8192 x 6144 x 4096 2808
// against 2733 (there the rounds fit).
struct TileUnits {
  double fixed, per_64_rows;
};
constexpr TileUnits TILE_UNITS{0.8, 0.8};
constexpr TileUnits TILE_UNITS_F32{0.1, 0.975};
inline double tile_cost_units(int mt, TileUnits u = TILE_UNITS) {
  return u.fixed + u.per_64_rows * mt;
}

// Relative cost of covering M x N with tiles of 64*mt rows on `cus` compute units: rounds of
// workgroups times the cost of one tile; shorter tiles re-read B more often per flop.
inline double tile_plan_cost(int64_t M, int64_t N, int mt, int cus, TileUnits u = TILE_UNITS) {
  const int64_t tiles = ((M + 64 * mt - 1) / (64 * mt)) * ((N + BN - 1) / BN);
  return (double)((tiles + cus - 1) / cus) * tile_cost_units(mt, u);
}
inline int best_mt(int64_t M, int64_t N, int cus, double* cost = nullptr,
                   TileUnits u = TILE_UNITS) {
  int best = 0;
  double bc = 1e30;
  for (int mt : {4, 3, 2, 1}) {
    const double c = tile_plan_cost(M, N, mt, cus, u);
    if (c < bc) {
      bc = c;
      best = mt;
    }
  }
  if (cost) *cost = bc;
  return best;
}

// The plan of a problem of more than one round of 256-row tiles.  When the tiles of the last round
// would leave much of the chip idle: the columns that fill whole rounds of 256-row tiles first
// (`first_cols` > 0), the remaining columns as a second, separately planned launch (which may split
// K).  Measured over 80 shapes with 5..24 row tiles (M = 1280..6144, N = 4096..14336; bf16 and int8
// N x K), the two launches issued from the host: where this rule takes them +3..+22 % (1536 x 11008 x
// 4096 bf16 143 -> 117 us, 3584 x 14336 x 4096 347 -> 314), at worst -3 %; the shapes it leaves alone
// would lose up to 7 %.
struct RoundsPlan {
  int mt;              // tile height of the one launch, or of the second when that is unsplit
  int64_t first_cols;  // columns of the first launch, 0: one launch
};
inline RoundsPlan plan_rounds(int64_t M, int64_t N, int cus, TileUnits units) {
  double single = 0;
  RoundsPlan r{best_mt(M, N, cus, &single, units), 0};
  const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  if (tiles_m > cus) return r;
  const int64_t cols_per_round = cus / tiles_m;
  const int64_t full_cols = (tiles_n / cols_per_round) * cols_per_round;
  if (full_cols <= 0 || full_cols >= tiles_n) return r;
  const int64_t n1 = full_cols * BN;
  double rest = 0;
  const int mt2 = best_mt(M, N - n1, cus, &rest, units);
  // (a tie stays with the single launch: int8 2048 x 11008 x 4096, 473 tiles of 192 rows in two
  // rounds against 256 tiles of 256 rows + 176 of 128 rows, alternating in one process: 85.3
  // against 86.0 us)
  if (tile_plan_cost(M, n1, 4, cus, units) + rest < single * 0.97) r = RoundsPlan{mt2, n1};
  return r;
}

// The height of a single launch of fp32 tiles: best_mt's choice among every multiple of 32 rows but 32.
inline int best_rows32(int64_t M, int64_t N, int cus, TileUnits u, double* cost) {
  const int64_t tiles_n = (N + BN - 1) / BN;
  int best = 0;
  *cost = 1e30;
  for (int rows = 256; rows >= 64; rows -= 32) {
    const int64_t tiles = (M + rows - 1) / rows * tiles_n;
    const double c = (double)((tiles + cus - 1) / cus) * (u.fixed + u.per_64_rows * rows / 64);
    if (c < *cost) *cost = c, best = rows;
  }
  return best;
}

// fp32: plan_rounds with every multiple of 32 rows (but 32) for the single launch, whose height goes to
// *rows; the second launch, which may split K, priced by the share of the chip its 64-row tiles take
// (4095 x 4097 x 4099: 17th column of tiles 63 us + 5 for the reduction, a quarter of a 64-row round
// is 60).  us before -> here: 20000 x 512 x 784 143.5 (210 tiles of 192 rows) -> 130.3 (250 of 160, one
// round), 3000^3 503 (192) -> 422 (160), 7000 x 4096 x 4096 1604 (64) -> 1588 (224).
// A second launch of more than 64 columns costs 0.35 units and 1 us beside its tiles: its ramp, its epilogue,
// the units that wait for the first one's last tiles (0.48 units below K = 64, where nothing was timed).
// 136 sizes where both plans were timed, K 64..4096, against the faster plan of each: 0.13 % slower on
// average, without that price 2.6 % (2111 x 8128 x 192 74.5 us in two launches, 65.5 in one of 96-row tiles;
// 2609 x 8160 x 64 47.6 and 43.9; 3188 x 7040 x 192 89.0 and 85.4).  Up to 64 columns end sooner, here or in
// kwaves_rest_columns.
inline RoundsPlan plan_rounds32(int64_t M, int64_t N, int64_t K_bytes, int cus, int* rows) {
  constexpr TileUnits u = TILE_UNITS_F32;
  const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  double best = 0;
  *rows = best_rows32(M, N, cus, u, &best);
  if (tiles_m > cus) return RoundsPlan{*rows / 64, 0};
  const int64_t cols_per_round = cus / tiles_m;
  const int64_t full_cols = tiles_n / cols_per_round * cols_per_round;
  if (full_cols <= 0 || full_cols >= tiles_n) return RoundsPlan{*rows / 64, 0};
  double rest = 0;
  const int mt2 = best_mt(M, N - full_cols * BN, cus, &rest, u);
  // (us of a unit: 64 rows of a tile over all stages of k)
  const double unit_us = STAGE_COST_KN32.per_64_rows_us * (double)((K_bytes + KB - 1) / KB);
  const double price = unit_us > 2.5 ? 0.35 + 1.0 / unit_us : 0.48;
  const double second = N - full_cols * BN > 64 ? price : 0.0;
  if (tiles_m * (tiles_n - full_cols) <= cus) {
    const double share =
        0.05 + (double)((M + 63) / 64 * (tiles_n - full_cols)) / cus * tile_cost_units(1, u);
    if (share < rest) rest = share;
  }
  if (tile_plan_cost(M, full_cols * BN, 4, cus, u) + rest + second < best)
    return RoundsPlan{mt2, full_cols * BN};
  return RoundsPlan{*rows / 64, 0};
}

}  // namespace tile
}  // namespace cig
