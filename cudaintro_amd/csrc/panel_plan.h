// Which calls the kernel of batches (gemm_panel.hip) takes and with tiles of how many rows, as plain host
// functions of sizes.
#pragma once
#include "any_plan.h"

namespace cig {
namespace panel {

constexpr int TN = 64, PB = 128;  // columns of a tile; bytes of k per stage

// us of one round of tiles: start, per stage, per stage and 64 rows, per 64 rows (the sums' meeting and the
// stores), per stage and 64 rows or columns of all units' tiles, operand bytes and output by the MB, int8 with
// scales.  Fitted to the kernel timed at 679 (16-bit) and 459 (int8) plans of sizes M 33..2048, N 256..16384, K
// 512..16384, log-uniform; rms error 6 and 8 %.
struct Cost {
  double start, stage, stage_64, tile_64, fetch, b_mb, a_mb, out_mb, dequant;
};
constexpr Cost COST_16{3.61, 0.156, 0.0593, 0.56, 0.0198, 0.0492, 0.157, 0.0, 0.0};
constexpr Cost COST_I8_NK{2.61, 0.138, 0.0707, 1.15, 0.0119, 0.0688, 0.219, 0.0663, 1.19};

inline double us(const Cost& c, const any::Problem& p, int cus, int rows) {
  const double stages = (double)any::div_up(p.K_bytes, PB), mt = rows / 64;
  const double share = (double)(any::div_up(p.M, rows) * any::div_up(p.N, TN)) / cus;
  return c.start + stages * (c.stage + c.stage_64 * mt + c.fetch * (mt + 1) * share) + c.tile_64 * mt +
         ((double)p.N * c.b_mb + (double)p.M * c.a_mb) * (double)p.K_bytes * 1e-6 +
         (double)p.M * (double)p.N * p.out_bytes * 1e-6 * c.out_mb + (p.dequant ? c.dequant : 0.0);
}

// Rows of a tile, 0: no call of this kernel's.  One round of tiles only, and sizes inside the timed ones.  Below
// 1536 bytes of k the estimates err too much (int8 641 x 2832 x 704 10.3 us here, 7.9 on the tile kernel); beyond
// 6000 the other one is often too high (int8 150 x 7040 x 10560 estimated 46 us there, took 38, here 47), and this
// one has to be 10 % below it.  Of some 2000 random calls that the tile kernel served with k up to 6000 bytes, 179
// 16-bit and 101 int8 ones are taken: 1.13 and 1.24 times as fast (geometric mean), 271 of them by more than 3 %,
// one more than 3 % slower (f16 67 x 13936 x 2544: 27.2 us, 23.9 there).  Of 316 taken among random sizes timed
// afterwards, 1.13 (16-bit) and 1.20 (int8) times as fast, five are 4 to 8 % slower.
inline int choose(const Cost& c, const any::Cost& other, const any::Problem& p, int cus, size_t partial_bytes) {
  if (p.M <= 32 || p.M > 2048 || p.N < 256 || p.K_bytes < 1536) return 0;
  int rows = 0;
  double best = 1e30;
  for (int r : {64, 128}) {
    if (r > 64 && p.M <= 64) break;
    if (any::div_up(p.M, r) * any::div_up(p.N, TN) > cus) continue;
    const double t = us(c, p, cus, r);
    if (t < best) best = t, rows = r;
  }
  if (p.K_bytes > 6000) best *= 1.1;
  return rows && best < any::other_us(other, p, true, cus, partial_bytes) ? rows : 0;
}

}  // namespace panel
}  // namespace cig
