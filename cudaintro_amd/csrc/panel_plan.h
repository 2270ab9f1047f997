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
// 1536 bytes of k the estimates err too much (int8 641 x 2832 x 704 10.3 us here, 7.9 on the tile kernel).  Beyond
// 5000 this one is often too low and the other too high (bf16 1860 x 720 x 2768 estimated 20.5 and 21.5 us, took 24.5
// and 21.3): it has to be 10 % below there, 2 % elsewhere.  Beyond 12000 two of 22 calls
// timed were faster by more than 3 % (5 and 7 %) and some far slower (int8 216 x 6464 x 13328 71 us, 54 there).  Of 2173 random calls with both
// estimates near or in favour, each timed on both kernels in turn, 1626 are taken: 1.18 times as fast
// (geometric mean), 1553 of them by more than 3 %, six more than 3 % slower (the worst 8 %); 32 were with one line
// at 6000 and no margin below it.  Of 1666 taken among as many random calls timed
// afterwards 1.18 times as fast, four more than 3 % slower (the worst 10 %).
inline int choose(const Cost& c, const any::Cost& other, const any::Problem& p, int cus, size_t partial_bytes) {
  if (p.M <= 32 || p.M > 2048 || p.N < 256 || p.K_bytes < 1536 || p.K_bytes > 12000) return 0;
  int rows = 0;
  double best = 1e30;
  for (int r : {64, 128}) {
    if (r > 64 && p.M <= 64) break;
    if (any::div_up(p.M, r) * any::div_up(p.N, TN) > cus) continue;
    const double t = us(c, p, cus, r);
    if (t < best) best = t, rows = r;
  }
  best *= p.K_bytes > 5000 ? 1.1 : 1.02;
  return rows && best < any::other_us(other, p, true, cus, partial_bytes) ? rows : 0;
}

}  // namespace panel
}  // namespace cig
