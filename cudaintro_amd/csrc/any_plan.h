// Which kernel serves a call of any size and alignment, as plain host functions of sizes (a host-only
// test checks them): the tile kernel's any-alignment form (gemm_any_tile.hip), the register-staged
// kernel (gemm_ragged.hip) or, fp32, the small kernel (gemm_f32_small.hip).
//
// The tile form has the higher rate and the higher price of a workgroup: tiles of 256 columns and
// at least 64 rows, K ranges of at least 8 stages, each stage a trip to memory before the first
// multiply, an epilogue through LDS.  So it loses where little of a tile is used or K is short: fp32
// 281391 x 11 x 16 105 us against 20 on the register-staged kernel, int8 4456 x 7 x 1575 21.9 against
// 11.8, bf16 33 x 11 x 741 13.7 against 9.2; and wins elsewhere: bf16 4096 x 4095 x 4096 111 against
// 264, fp32 4095 x 4097 x 4099 979 against 1499.  Both estimates below have the terms that decide
// between them; their constants were fitted to the kernels timed at 850 sizes of each 16-bit and int8
// layout and 1570 of fp32 (M 1..300000, N 2..16384, K 16..16384, log-uniform, packed, few of them
// aligned).  The kernel chosen by them was 0.4 % (16-bit), 0.5 and 0.9 % (int8 K x N, N x K) and 0.3 %
// (fp32) slower than the fastest on average; the tile form wherever it is possible 5..6 % and (fp32)
// 56 %, the register-staged kernel throughout 21..24 % and 53 % (profiles/any_kernel_choice.md).
#pragma once
#include "tile_plan.h"

namespace cig {
namespace any {

struct Problem {
  int64_t M, N, K_bytes;
  int elem, out_bytes;
  bool dequant;       // int8 with scales
  bool a_apart, b_apart;  // rows of that operand do not all start at multiples of 4 bytes
};

// us; *_mb per 1e6 bytes
struct Cost {
  // tile form: start + rounds x (stages x (stage + stage_64_rows x rows / 64 + apart x 64-row pieces
  // of operand tiles that the address path takes apart) + tile_64_rows x rows / 64) + traffic + a
  // share of the planner's price of the reduction, summed over the launches of the plan
  double t_start, t_stage, t_stage_64_rows, t_apart, t_tile_64_rows, t_out_mb, t_in_mb, t_reduce,
      t_dequant;
  // register-staged kernel: start + steps per range x (step + step_unit x workgroups per unit, rounded up) +
  // traffic + reduction; its epilogue is element by element, dearer with rows to fill it (s_rows)
  // and with scales (s_dequant, unsplit only: else the reduction applies them)
  double s_start, s_step, s_step_unit, s_out_mb, s_reduce, s_reduce_mb, s_rows, s_dequant,
      s_dequant_mb, s_in_mb;
  tile::StageCost sc;
  tile::TileUnits units;
};
constexpr Cost COST_16{
    4.23, 0.0346, 0.125, 0.0273, 1.24, 0.129, 0.0661, 0.689, 0.0,
    4.56, 0.195, 0.363, 0.222, 3.16, 0.097, 0.0862, 0.0, 0.0, 0.01,
    tile::STAGE_COST_KN16, tile::TILE_UNITS};
constexpr Cost COST_F32{
    2.62, 0.153, 0.799, 0.0, 2.73, 0.0775, 0.0692, 0.538, 0.0,
    4.24, 0.312, 1.04, 0.15, 2.93, 0.203, 0.0, 0.0, 0.0, 0.0249,
    tile::STAGE_COST_KN32, tile::TILE_UNITS_F32};
constexpr Cost COST_I8_KN{
    4.48, 0.0687, 0.112, 0.043, 1.76, 0.116, 0.0653, 0.44, 0.599,
    5.56, 0.118, 0.411, 0.15, 3.31, 0.18, 0.0126, 5.3, 0.449, 0.0,
    tile::STAGE_COST_KN8, tile::TILE_UNITS};
constexpr Cost COST_I8_NK{
    4.84, 0.0533, 0.126, 0.0361, 1.34, 0.136, 0.0991, 0.518, 0.704,
    5.79, 0.0191, 0.447, 0.165, 3.14, 0.151, 1.02, 3.28, 0.433, 0.0,
    tile::STAGE_COST_NK8, tile::TILE_UNITS};

inline int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }
// (see Problem::a_apart)
inline bool rows_apart(const void* p, int64_t ld_bytes) {
  return (((uintptr_t)p | (uintptr_t)ld_bytes) & 3) != 0;
}
inline double at_most(double v, double top) { return v < top ? v : top; }

// What the tile form takes: sizes only.  One 16-byte piece must fit a row of either operand (and a
// column of k); the launch-size and 32-bit offset limits are the aligned form's.
inline bool tile_ok(int64_t M, int64_t N, int64_t K, int elem, int64_t lda, int64_t ldb, bool b_kn) {
  if (M <= 0 || N <= 0 || K * elem < 16 || (b_kn && N * elem < 16)) return false;
  if (M > 2147483647LL - 255 || N > 2147483647LL - 255 || K * elem > 2147483647LL) return false;
  if (((M + 63) / 64) * ((N + tile::BN - 1) / tile::BN) > 2147483647LL) return false;
  return lda * elem * 256 < (1LL << 31) && ldb * elem * 256 < (1LL << 31);
}

// The any-alignment form's plan when at most one round of 256-row tiles covers the output (mt = 0:
// more than that, the launcher then plans by rounds).  Partial sums have rows of whole lines.
inline tile::SmallPlan tile_plan(const Cost& c, const Problem& p, int cus, size_t partial_bytes) {
  if (div_up(p.M, tile::BM) * div_up(p.N, tile::BN) > cus) return tile::SmallPlan{0, 1};
  return tile::plan_small(cus, partial_bytes, p.M, div_up(p.N, 32) * 32, p.K_bytes, p.out_bytes, c.sc,
                          p.K_bytes * p.N);
}

// Rows of the tiles that the launcher runs `plan` of N columns with: fp32 may have a height between.
inline int tile_rows(const Cost& c, const Problem& p, int64_t N, int cus, tile::SmallPlan plan) {
  return p.elem == 4 ? tile::plan_small_rows32(cus, p.M, N, p.K_bytes, p.out_bytes, c.sc, p.K_bytes * N,
                                               plan)
                     : 64 * plan.mt;
}

// One launch of the tile form (and the reduction behind it): N columns on tiles of `rows` rows.
inline double tile_launch_us(const Cost& c, const Problem& p, int64_t N, int cus, int rows, int splits) {
  const double mt = rows / 64.0;
  int64_t stages = 0;
  const int sp = tile::k_ranges(p.K_bytes, splits, &stages);
  const double rounds = (double)div_up(div_up(p.M, rows) * div_up(N, tile::BN) * sp, cus);
  const double apart = (p.a_apart ? mt : 0) + (p.b_apart ? 4 : 0);
  const double mn = (double)p.M * (double)N * 1e-6;
  double us = rounds * ((double)stages * (c.t_stage + c.t_stage_64_rows * mt + c.t_apart * apart) +
                        c.t_tile_64_rows * mt);
  us += c.t_out_mb * mn * (sp > 1 ? sp * 4 : p.out_bytes) +
        c.t_in_mb * (double)(p.M + N) * (double)p.K_bytes * 1e-6;
  if (sp > 1) {
    const double reduce = 1.1 + (sp * 4 + p.out_bytes) * mn / 5.3;
    us += c.t_reduce * (reduce > 4.75 ? reduce : 4.75);
  }
  return us;
}

inline double tile_us(const Cost& c, const Problem& p, int cus, size_t partial_bytes,
                      tile::SmallPlan plan) {
  const double us = c.t_start + (p.dequant ? c.t_dequant : 0.0);
  if (plan.mt) return us + tile_launch_us(c, p, p.N, cus, tile_rows(c, p, p.N, cus, plan), plan.splits);
  int rows = 0;
  tile::RoundsPlan r;
  if (p.elem == 4) {
    r = tile::plan_rounds32(p.M, p.N, p.K_bytes, cus, &rows);
  } else {
    r = tile::plan_rounds(p.M, p.N, cus, c.units);
    rows = 64 * r.mt;
  }
  if (!r.first_cols) return us + tile_launch_us(c, p, p.N, cus, rows, 1);
  Problem rest = p;
  rest.N = p.N - r.first_cols;
  const tile::SmallPlan second = tile_plan(c, rest, cus, partial_bytes);
  return us + tile_launch_us(c, p, r.first_cols, cus, 256, 1) +
         tile_launch_us(c, rest, rest.N, cus,
                        second.mt ? tile_rows(c, rest, rest.N, cus, second) : 64 * r.mt, second.splits);
}

// K ranges of the register-staged kernel (tiles of 128 x 128, steps of 64 bytes of k) for a problem
// of few tiles, a decode or small-batch shape: about three workgroups per compute unit are resident,
// so enough ranges to fill those places, each of at least four steps, at most 16, partials within
// the workspace.  bf16 N = 8191, K = 8192, M = 1 (64 tiles): 255 us unsplit, 31.5 split.
// `range_steps` receives the steps of each range but the last.
inline int staged_ranges(const Problem& p, int cus, size_t partial_bytes, int64_t* range_steps) {
  const int64_t tiles = div_up(p.M, 128) * div_up(p.N, 128), steps = div_up(p.K_bytes, tile::KB);
  int64_t s = 1;
  if (partial_bytes && tiles * 2 <= 3 * (int64_t)cus) {  // (two ranges fit)
    s = 3 * (int64_t)cus / tiles;
    if (s > 16) s = 16;
    if (s > steps / 4) s = steps / 4;
    while (s > 1 && (size_t)s * (size_t)p.M * (size_t)p.N * 4 > partial_bytes) --s;
    if (s < 1) s = 1;
  }
  *range_steps = div_up(steps, s);
  return steps > 0 ? (int)div_up(steps, *range_steps) : 1;  // ranges that would start past K go
}

inline double staged_us(const Cost& c, const Problem& p, int cus, size_t partial_bytes) {
  int64_t steps = 0;
  const int sp = staged_ranges(p, cus, partial_bytes, &steps);
  const double per = (double)div_up(div_up(p.M, 128) * div_up(p.N, 128) * sp, cus);
  const double mn = (double)p.M * (double)p.N * 1e-6, rows = at_most((double)p.M / 128, 1.0);
  double us = c.s_start + (double)steps * (c.s_step + c.s_step_unit * per);
  us += c.s_out_mb * mn * (sp > 1 ? sp * 4 : p.out_bytes) +
        c.s_in_mb * (double)(p.M + p.N) * (double)p.K_bytes * 1e-6 + c.s_rows * rows;
  if (sp > 1) us += c.s_reduce + c.s_reduce_mb * mn * (4 * sp + p.out_bytes);
  if (p.dequant) us += (sp > 1 ? 0.0 : c.s_dequant * rows) + c.s_dequant_mb * mn;
  return us;
}

// What the tile kernel or the register-staged kernel is estimated to take, whichever serves the call;
// `aligned`: the tile kernel's aligned form does (the same terms rank it: rms error 12..14 % over
// 250 aligned calls).
inline double other_us(const Cost& c, const Problem& p, bool aligned, int cus, size_t partial_bytes) {
  if (aligned) {
    tile::SmallPlan plan{0, 1};
    if (div_up(p.M, tile::BM) * div_up(p.N, tile::BN) <= cus)
      plan = tile::plan_small(cus, partial_bytes, p.M, p.N, p.K_bytes, p.out_bytes, c.sc,
                              p.K_bytes * p.N);
    return tile_us(c, p, cus, partial_bytes, plan);
  }
  const double staged = staged_us(c, p, cus, partial_bytes);
  const double tile = tile_us(c, p, cus, partial_bytes, tile_plan(c, p, cus, partial_bytes));
  return staged < tile ? staged : tile;
}

// The small fp32 kernel: 32 x 32 tiles, K walked by four waves, so a chain of loads whose price
// per k depends on how many tiles share a unit and on whether B's rows are read in 16-byte pieces
// (`b16`); or, `narrow`, its 16 x 16 form, which streams A.
inline double f32_small_us(int64_t M, int64_t N, int64_t K, int cus, bool b16, bool narrow) {
  const double m = (double)M, n = (double)N, k = (double)K;
  if (narrow) {
    const int64_t blocks = (K / 16 + 3) / 4;  // of a wave; the kernel comes for 8, 16 or 32
    const double form = blocks <= 8 ? 8.0 : blocks <= 16 ? 16.0 : 32.0;
    return 1.85 + 0.18e-6 * 4.0 * m * k + 0.348 * (double)blocks +
           0.123 * form * (double)div_up(div_up(M, 16), 4 * (int64_t)cus);
  }
  const int64_t tiles = div_up(M, 32) * div_up(N, 32), rounds = div_up(tiles, cus);
  const double mb = (m + n) * k * 4e-6;  // of both operands, against the caches' reach
  const double per_k =
      rounds > 1 ? ((b16 ? 0.00656 : 0.00775) + 0.00195 * at_most(mb / 256.0, 1.0)) * (double)rounds
                 : 0.0061 + 0.00196 * (double)tiles / cus + 0.00542 * at_most(mb / 27.5, 1.0);
  return 2.5 + k * per_k + 0.223e-6 * 4.0 * m * n + 0.071 * (double)rounds;
}

}  // namespace any
}  // namespace cig
