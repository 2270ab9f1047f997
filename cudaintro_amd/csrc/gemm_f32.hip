// fp32 GEMM on the gfx950 matrix cores (v_mfma_f32_32x32x2_f32: fp32 products, fp32
// accumulation): the shared LDS-tiled MFMA kernel with the fp32 fragment plumbing, plain or
// with the linear layer's bias + activation epilogue; or, when 256-column tiles would leave
// most of the chip idle or N is too ragged for them, the 32x32 k-split kernel.
#include "any_plan.h"
#include "epilogues.h"
#include "mfma_tile.h"

namespace cig {

bool f32_tile_ok(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                        const float* B, int64_t ldb, const float* C, int64_t ldc,
                        const BiasAct* ba) {
  return tile::tile_shape_ok(M, N, K, 4, A, lda, B, ldb, true) && ldc % 4 == 0 &&
         ((uintptr_t)C & 15) == 0 && !(ba && ba->bias && ((uintptr_t)ba->bias & 15));
}

// Whether a call that the tile kernel takes is the small kernel's.
static bool aligned_is_small(const cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A,
                             int64_t lda, const float* B, int64_t ldb) {
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const bool one_round = ((M + 255) / 256) * ((N + tile::BN - 1) / tile::BN) <= cus;
  if (f32_small_shape_ok(M, N, K, A, lda)) {
    // Both costs in units of a quarter of one 256x256 tile's time per unit of k: the tile
    // plan's own figure against 0.115 per resident round of 32x32 tiles (2048^3: tile kernel
    // 157 us, small kernel 225 us; 1024^3: 74 us against 33 us; 512^3: 38 us against 8 us).
    double tile_cost = 0;
    tile::best_rows32(M, N, cus, tile::TILE_UNITS, &tile_cost);
    const double tiles32 = (double)((M + 31) / 32) * (double)((N + 31) / 32);
    const double small_cost = 0.115 * (tiles32 > cus ? tiles32 / cus : 1.0);
    // With a long K the tile kernel wins whenever its tiles fit one round: it can split K over
    // the idle compute units (512 x 512 x 4096: 33 us against 55 us; 1024^3: 31 against 32;
    // 512^3: 17 against 9; 960 x 3584 x 3584: 222 against 298).
    return small_cost < tile_cost && !(K >= 2048 && one_round);
  } else if (f32_small_any_ok(M, N, K)) {
    // A K of whole 16-byte pieces that is no multiple of 8: by the small kernel's estimate against
    // the planner's + 4 us, or against what the launches of several rounds are estimated at.  Over
    // 300 sizes 0.5 % slower than the faster of the two on average; the tile kernel throughout 38 %,
    // the comparison above 1.8 %: 3837 x 808 x 1588 144 us on the small kernel against 100, 78 x 1900
    // x 1972 25.6 against 19.9.
    const size_t room = ctx->workspace ? ctx->ws_partial_bytes : 0;
    double tile_us = 0;
    if (one_round) {
      const tile::SmallPlan plan =
          tile::plan_small(cus, room, M, N, K * 4, 4, tile::STAGE_COST_KN32, K * 4 * N);
      tile::plan_small_rows32(cus, M, N, K * 4, 4, tile::STAGE_COST_KN32, K * 4 * N, plan, &tile_us);
      tile_us += 4.0;
    } else {
      tile_us = any::tile_us(any::COST_F32, any::Problem{M, N, K * 4, 4, 4, false, false, false}, cus,
                             room, tile::SmallPlan{0, 1});
      // (that is the any-alignment form; a K of one stage is a single trip here, there a tail and a
      // loop: 81708 x 356 x 12 38.3 us, estimated 48.0, small kernel 54.4)
      if (K <= 16) tile_us *= 0.73;
    }
    return any::f32_small_us(M, N, K, cus, f32_small_b16(N, B, ldb), false) < tile_us;
  }
  return false;
}

bool launch_f32_mfma(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A,
                     int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                     const BiasAct* ba) {
  if (!f32_tile_ok(M, N, K, A, lda, B, ldb, C, ldc, ba)) return false;
  if (!aligned_is_small(ctx, M, N, K, A, lda, B, ldb))
    return launch_f32_tile(ctx, M, N, K, A, lda, B, ldb, C, ldc, ba);
  launch_f32_small(ctx, M, N, K, A, lda, B, ldb, C, ldc, ba);
  return true;
}

F32Other f32_other(const cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A,
                   int64_t lda, const float* B, int64_t ldb, const float* C, int64_t ldc,
                   const BiasAct* ba) {
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const size_t room = ctx->workspace ? ctx->ws_partial_bytes : 0;
  const any::Problem p{M, N, K * 4, 4, 4, false, false, false};
  const F32Other small{
      f32_small_any_ok(M, N, K) ? any::f32_small_us(M, N, K, cus, f32_small_b16(N, B, ldb),
                                                    f32_small_is_narrow(M, N, K, A, lda))
                                : 1e30,
      any::div_up(K, 4), true};
  if (f32_tile_ok(M, N, K, A, lda, B, ldb, C, ldc, ba)) {
    if (aligned_is_small(ctx, M, N, K, A, lda, B, ldb)) return small;
    tile::SmallPlan plan{0, 1};
    if (any::div_up(M, tile::BM) * any::div_up(N, tile::BN) <= cus)
      plan = tile::plan_small(cus, room, M, N, K * 4, 4, any::COST_F32.sc, K * 4 * N);
    return F32Other{any::tile_us(any::COST_F32, p, cus, room, plan), K / plan.splits, false};
  }
  const tile::SmallPlan plan = any::tile_plan(any::COST_F32, p, cus, room);
  const double tile = any::tile_us(any::COST_F32, p, cus, room, plan);
  const double staged = any::staged_us(any::COST_F32, p, cus, room);
  int64_t steps = 0;
  const F32Other other = staged < tile ? F32Other{staged, K / any::staged_ranges(p, cus, room, &steps), false}
                                       : F32Other{tile, K / plan.splits, false};
  return small.us < other.us ? small : other;
}

bool launch_f32_tile(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A,
                     int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                     const BiasAct* ba) {
  if (!f32_tile_ok(M, N, K, A, lda, B, ldb, C, ldc, ba)) return false;
  if (!ba) {
    const bool split = tile::launch_tile<tile::MathF32, tile::B_KN32>(
        ctx, M, N, K * 4, A, lda * 4, B, ldb * 4, EpiStoreF32x4{C, ldc});
    set_tile_kernel_name(ctx, "f32", 16, "_32x32x2", split);
    return true;
  }
  bool split = false;
#define CIG_BA(HB, RL)                                                                          \
  split = tile::launch_tile<tile::MathF32, tile::B_KN32>(ctx, M, N, K * 4, A, lda * 4, B, ldb * 4, \
                                                         EpiBiasActF32x4<HB, RL>{C, ldc, ba->bias})
  if (ba->bias) {
    if (ba->relu) CIG_BA(true, true); else CIG_BA(true, false);
  } else {
    if (ba->relu) CIG_BA(false, true); else CIG_BA(false, false);
  }
#undef CIG_BA
  set_tile_kernel_name(ctx, "f32", 16, "_32x32x2_bias_act", split);
  return true;
}

}  // namespace cig
