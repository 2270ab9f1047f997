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

constexpr int TM = 32, TN = 64, PB = 128;  // output tile; bytes of k per piece
constexpr int WAVES = 4;

// The plan's grid fits a launch, and its partial sums and arrival counters their parts of the
// workspace.
inline bool fits(int64_t M, int64_t N, Plan p, size_t partial_bytes, size_t counter_bytes) {
  const int64_t tiles = any::div_up(M, TM) * any::div_up(N, TN);
  if (tiles > 2147483647LL / p.splits) return false;
  return p.splits == 1 || (tiles <= (int64_t)(counter_bytes / 4) &&
                           tiles * p.splits * TM * TN * 4 <= (int64_t)partial_bytes);
}

// us: a call's start, then per piece of the workgroups that share the fullest compute unit (what the
// unit takes from its L2), per piece on average (what the chip takes from memory), per workgroup of
// that unit; pieces the address path takes apart, operand bytes, and for K ranges their meeting and
// the bytes of their sums.  Fitted to the kernel timed at 320 sizes of each layout (M 17..3000, N and
// K 64..16384, log-uniform, 40 % of the widths odd) x up to 8 numbers of ranges; rms error 9..12 %.
struct Cost {
  double start, unit_piece, load, unit_tile, apart, in_mb, split, part_mb, tail, dequant;
};
constexpr Cost COST_16{3.95, 0.0849, 0.0562, 0.0155, 0.0202, 0.0664, 1.46, 0.130, 1.05, 0.0};
constexpr Cost COST_I8_KN{4.31, 0.0907, 0.103, 0.0, 0.0342, 0.0608, 1.32, 0.0941, 0.365, 0.692};
constexpr Cost COST_I8_NK{4.47, 0.0708, 0.0599, 0.0990, 0.0299, 0.0759, 1.09, 0.163, 0.552, 0.717};

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
  return est < any::other_us(other, p, aligned, cus, partial_bytes) ? b : Plan{0};
}

}  // namespace kwaves
}  // namespace cig
