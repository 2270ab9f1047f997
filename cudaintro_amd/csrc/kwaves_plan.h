// Launch planning of the kernel of small outputs (gemm_kwaves.hip), as plain host functions of sizes:
// the number of K ranges, and whether the kernel is estimated to be faster than what would serve the
// call otherwise.
#pragma once
#include "any_plan.h"

namespace cig {
namespace kwaves {

struct Plan {
  int splits;  // K ranges; 0: no plan
};

constexpr int TM = 32, TN = 64, PB = 128;  // output tile (fp32: 32 columns); bytes of k per piece
constexpr int WAVES = 4;

// The plan's grid fits a launch, and its partial sums and arrival counters their parts of the
// workspace.
inline bool fits(int64_t M, int64_t N, Plan p, size_t partial_bytes, size_t counter_bytes,
                 int tn = TN) {
  const int64_t tiles = any::div_up(M, TM) * any::div_up(N, tn);
  if (tiles > 2147483647LL / p.splits) return false;
  return p.splits == 1 || (tiles <= (int64_t)(counter_bytes / 4) &&
                           tiles * p.splits * TM * tn * 4 <= (int64_t)partial_bytes);
}

// us: a call's start, then per piece of the workgroups that share the fullest compute unit (what the
// unit takes from its L2), per piece on average (what the chip takes from memory), per workgroup of
// that unit; pieces the address path takes apart, operand bytes, and for K ranges their meeting and
// the bytes of their sums.  Fitted to the kernel timed at 320 sizes of each layout (M 17..3000, N and
// K 64..16384, log-uniform, 40 % of the widths odd) x up to 8 numbers of ranges; rms error 9..12 %.
// Long streams of k, where that is too low: the estimate has to win by 30 % (N x K) or 10 % (K x N) there.
// N x K: 65 to 768 columns whose k is no whole pieces, once a unit takes more than 8000 bytes of k for all
// of its workgroups (787 x 392 x 15048 29.8 us here, 22.1 on the tile kernel; 8748 x 72 x 6000 35.4 and
// 26.5; with whole pieces 387 x 1066 x 12416 16.7 and 20.8).  K x N: rows of more than 128 bytes, ranges of more
// than `long_range` bytes that at least half of the units have (bf16 904 x 276 x 3896 17.6 and 14.1, 757 x
// 570 x 3856 18.3 and 15.9; of narrower outputs int8 3615 x 99 x 5552 16.2 and 20.3).  Of 11468 random
// sizes taken before, most of them with 120..768 tiles, 637 were more than 3 % slower here than without
// this kernel, 195 of those taken now; 56 that were more than 3 % faster are taken no longer.
struct Cost {
  double start, unit_piece, load, unit_tile, apart, in_mb, split, part_mb, tail, dequant;
  double long_range;  // bytes; 0: N x K
};
constexpr Cost COST_16{3.95, 0.0849, 0.0562, 0.0155, 0.0202, 0.0664, 1.46, 0.130, 1.05, 0.0, 7000};
constexpr Cost COST_I8_KN{4.31, 0.0907, 0.103, 0.0, 0.0342, 0.0608, 1.32, 0.0941, 0.365, 0.692, 5000};
constexpr Cost COST_I8_NK{4.47, 0.0708, 0.0599, 0.0990, 0.0299, 0.0759, 1.09, 0.163, 0.552, 0.717, 0};

// `whole`: no tail (k and the rows of a K x N operand are whole pieces)
inline double us(const Cost& c, const any::Problem& p, bool whole, int cus, int splits) {
  int64_t stages = 0;
  const int sp = tile::k_ranges(p.K_bytes, splits, &stages);
  const int64_t pieces = any::div_up(stages, 2);
  const int64_t wgs = any::div_up(p.M, TM) * any::div_up(p.N, TN) * sp, per = any::div_up(wgs, cus);
  const double apart = (p.a_apart ? 1 : 0) + (p.b_apart ? 2 : 0);
  double t = c.start + (double)(per * pieces) * (c.unit_piece + c.apart * apart) +
             (double)wgs / cus * (double)pieces * c.load + (double)per * c.unit_tile +
             (double)(p.M + p.N) * (double)p.K_bytes * 1e-6 * c.in_mb + (whole ? 0.0 : c.tail) +
             (p.dequant ? c.dequant : 0.0);
  if (sp > 1) t += c.split + (double)p.M * (double)p.N * 4e-6 * sp * c.part_mb;
  return t;
}

// The best number of K ranges, each of at least 1 KiB of k (two pieces a wave); its estimate in *est.
inline Plan best(const Cost& c, const any::Problem& p, bool whole, int cus, size_t partial_bytes,
                 size_t counter_bytes, double* est) {
  Plan b{1};
  *est = us(c, p, whole, cus, 1);
  const int64_t tiles = any::div_up(p.M, TM) * any::div_up(p.N, TN);
  for (int sp = 2; sp <= 16 && p.K_bytes / sp >= 1024 && tiles * sp <= 4 * (int64_t)cus; ++sp) {
    if (!fits(p.M, p.N, Plan{sp}, partial_bytes, counter_bytes)) break;
    const double t = us(c, p, whole, cus, sp);
    if (t < *est) *est = t, b = Plan{sp};
  }
  return b;
}

// The plan, or no plan (0) where another kernel is estimated to be faster.  A K of no more than three
// pieces leaves waves without one, and the tile kernels are as fast there (bf16 646 x 6848 x 64 7.0 us
// against 9.8 here).  More tiles than are resident at once (three workgroups a unit) are the tile
// kernels' as well (int8 N x K 5129 x 384 x 960 8.7 against 12.2), and so are outputs of fewer than 16
// columns the register-staged kernel's.
inline Plan choose(const Cost& c, const any::Cost& other, const any::Problem& p, bool whole,
                   bool aligned, int cus, size_t partial_bytes, size_t counter_bytes) {
  const int64_t tiles = any::div_up(p.M, TM) * any::div_up(p.N, TN);
  if (p.K_bytes <= 3 * PB || p.N < 16 || tiles > 3 * (int64_t)cus) return Plan{0};
  double est = 0;
  const Plan b = best(c, p, whole, cus, partial_bytes, counter_bytes, &est);
  // (beyond one round the two estimates have to differ by more than they usually err)
  if (tiles > cus) est *= 1.1;
  int64_t stages = 0;
  const int sp = tile::k_ranges(p.K_bytes, b.splits, &stages);
  const double range = (double)p.K_bytes / sp;
  if (c.long_range > 0) {
    if (p.N * p.elem > PB && 2 * tiles > cus && range > c.long_range) est *= 1.1;
  } else if (!whole && p.N > TN && p.N <= 768 && (double)any::div_up(tiles * sp, cus) * range > 8000.0) {
    est *= 1.3;
  }
  return est < any::other_us(other, p, aligned, cus, partial_bytes) ? b : Plan{0};
}

// ---- fp32: tiles of 32 x 32 ---------------------------------------------------------------------
// us: `start`, then per piece of the busiest wave of a unit (its 16 matrix instructions: the unit's
// workgroups one after the other) and of a workgroup's busiest wave, per piece on average, per
// workgroup of a unit, operand bytes, K ranges and the tail.  Fitted to the kernel timed at 420 sizes
// (M 1..6000, N 4..8192, K 16..8192, log-uniform) x up to 8 numbers of ranges; rms error 7 %.
struct CostF32 {
  double start, unit_piece, wave_piece, load, unit_tile, in_mb, split, part_mb, tail;
};
constexpr CostF32 COST_F32{4.58, 0.341, 0.140, 0.0441, 0.123, 0.0160, 0.816, 0.107, 0.375};
constexpr int TN_F32 = 32;
// No range of k is longer than 64 pieces (2048 floats, 512 for each wave to add up): a long K keeps
// the rounding of the shorter sums it has on the tile kernel, and the ranges cost 0.8 us.
constexpr int MAX_RANGE_BYTES_F32 = 64 * PB;

inline double us_f32(int64_t M, int64_t N, int64_t K, int cus, int splits) {
  const CostF32& c = COST_F32;
  int64_t stages = 0;
  const int sp = tile::k_ranges(K * 4, splits, &stages);
  const int64_t pieces = any::div_up(stages, 2), wave = any::div_up(pieces, WAVES);
  const int64_t wgs = any::div_up(M, TM) * any::div_up(N, TN_F32) * sp, per = any::div_up(wgs, cus);
  double t = c.start + (double)(per * wave) * c.unit_piece + (double)wave * c.wave_piece +
             (double)wgs / cus * (double)pieces * c.load + (double)per * c.unit_tile +
             (double)(M + N) * (double)K * 4e-6 * c.in_mb + (K % 32 || N % 4 ? c.tail : 0.0);
  if (sp > 1) t += c.split + (double)M * (double)N * 4e-6 * sp * c.part_mb;
  return t;
}

// The plan with the lowest estimate, which goes to *est; no plan (0) for a K of no more than two pieces,
// more tiles than four a unit, a K of more ranges than 16, or operands beyond the 256 MB cache, whose
// stream the 256-column tiles keep up better (39 x 9664 x 9984 130 us against 116).
inline Plan best_f32(int64_t M, int64_t N, int64_t K, int cus, size_t partial_bytes,
                     size_t counter_bytes, double* est) {
  const int64_t tiles = any::div_up(M, TM) * any::div_up(N, TN_F32), K_bytes = 4 * K;
  const int64_t least = any::div_up(K_bytes, MAX_RANGE_BYTES_F32);
  *est = 1e30;
  Plan b{0};
  if (K_bytes <= 2 * PB || tiles > 4 * (int64_t)cus || (M + N) * K_bytes > 256000000) return b;
  for (int64_t sp = least; sp <= 16; ++sp) {
    if (sp > least && (K_bytes / sp < 1024 || tiles * sp > 4 * (int64_t)cus)) break;
    if (!fits(M, N, Plan{(int)sp}, partial_bytes, counter_bytes, TN_F32)) break;
    const double t = us_f32(M, N, K, cus, (int)sp);
    if (t < *est) *est = t, b = Plan{(int)sp};
  }
  // Where the estimate is too low, it has to be below the other by more.  Row tiles that share a B beyond
  // what the L2s keep: 20 % from 128 MB of it on (36 x 5016 x 7040 estimated 46 us, took 60; 45 on the
  // tile kernel; a long A is no such stream: 15963 x 8 x 1146 16.7 us here, 22.4 register-loaded).  Four to seven workgroups a unit, of which three are resident: 12 % (467 x 768 x 7936
  // 64 us, tile kernel 56), but for outputs of up to 128 columns, which the other kernels pad (7250 x 64 x
  // 5935 76 us here, 115 there).  Beyond a round and a half: 12 % (127 x 7360 x 4032 79 and 70, estimated
  // equal).  Of 1094 sizes around these lines that were taken before, 313 were more than 3 % slower here
  // than on the other kernels (the worst 29 %), 38 of those taken now; the choice is 0.6 % off the faster
  // kernel on average, 3.9 % before.
  const double mb = (double)N * (double)K_bytes * 1e-6;
  if (M > TM && mb > 48.0) *est *= 1.0 + 0.2 * any::at_most((mb - 48.0) / 80.0, 1.0);
  if (tiles * b.splits > 4 * (int64_t)cus && tiles * b.splits <= 7 * (int64_t)cus && N > 128) *est *= 1.12;
  if (2 * tiles > 3 * (int64_t)cus) *est *= 1.12;
  return b;
}

}  // namespace kwaves
}  // namespace cig
