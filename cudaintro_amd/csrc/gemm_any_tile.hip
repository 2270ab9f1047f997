// The LDS-DMA tile kernel at any alignment (mfma_tile.h, ANY): the calls whose sizes, leading
// dimensions or pointers the aligned form's gate turns away (an odd N, a K whose bytes are not a
// multiple of 16, rows or pointers that are not 16-byte aligned; the library this path replaces
// takes any m, n, k, lda, ldb: quantization/GEMM_bf16.cu:51-56).  Same plans -- tile heights, K
// ranges, two-launch form -- as the aligned calls; kernel names carry "_mfma_any_".
// int8 results equal the CPU loop bit for bit; the floating types are within the bounds of the
// aligned form (the last 1..64 bytes of k are summed first here).
#include "any_plan.h"
#include "epilogues.h"
#include "mfma_tile.h"

namespace cig {
namespace {

template <int BMODE>
bool launch_i8_layout(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const int8_t* A,
                      int64_t lda, const int8_t* B, int64_t ldb, int32_t* C, int64_t ldc,
                      const DequantArgs* dq, tile::SmallPlan plan) {
  if (!dq)
    return tile::launch_tile<tile::MathI8, BMODE, true>(ctx, M, N, K, A, lda, B, ldb,
                                                        EpiStoreI32x4{C, ldc}, plan);
  if (dq->out_bf16)
    return tile::launch_tile<tile::MathI8, BMODE, true>(
        ctx, M, N, K, A, lda, B, ldb,
        EpiDequantX4<true, false>{dq->out, dq->ldo, dq->sa, dq->sb, dq->sa_vec, dq->sb_vec,
                                  nullptr, 0},
        plan);
  return tile::launch_tile<tile::MathI8, BMODE, true>(
      ctx, M, N, K, A, lda, B, ldb,
      EpiDequantX4<false, false>{dq->out, dq->ldo, dq->sa, dq->sb, dq->sa_vec, dq->sb_vec, nullptr,
                                 0},
      plan);
}

}  // namespace

bool launch_tile_any_16(cigemmContext* ctx, bool bf16, int64_t M, int64_t N, int64_t K,
                        const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb,
                        uint16_t* C, int64_t ldc, tile::SmallPlan plan) {
  if (!any::tile_ok(M, N, K, 2, lda, ldb, true)) return false;
  if (bf16)
    set_tile_kernel_name(ctx, "bf16", 32, "",
                         tile::launch_tile<tile::MathBF16, tile::B_KN16, true>(
                             ctx, M, N, K * 2, A, lda * 2, B, ldb * 2, EpiStore16x4<BF16>{C, ldc},
                             plan),
                         true);
  else
    set_tile_kernel_name(ctx, "f16", 32, "",
                         tile::launch_tile<tile::MathF16, tile::B_KN16, true>(
                             ctx, M, N, K * 2, A, lda * 2, B, ldb * 2, EpiStore16x4<F16>{C, ldc},
                             plan),
                         true);
  return true;
}

bool launch_tile_any_f32(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A,
                         int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                         const BiasAct* ba, tile::SmallPlan plan) {
  if (!any::tile_ok(M, N, K, 4, lda, ldb, true)) return false;
  const bool split =
      ba ? tile::launch_tile<tile::MathF32, tile::B_KN32, true>(
               ctx, M, N, K * 4, A, lda * 4, B, ldb * 4,
               EpiBiasActAnyF32x4{C, ldc, ba->bias, ba->relu}, plan)
         : tile::launch_tile<tile::MathF32, tile::B_KN32, true>(ctx, M, N, K * 4, A, lda * 4, B,
                                                                ldb * 4, EpiStoreF32x4{C, ldc}, plan);
  set_tile_kernel_name(ctx, "f32", 16, ba ? "_32x32x2_bias_act" : "_32x32x2", split, true);
  return true;
}

// (the accumulator dump, a second output of every quad, is left to the older any-shape kernel)
bool launch_tile_any_i8(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const int8_t* A,
                        int64_t lda, const int8_t* B, int64_t ldb, bool b_nk, int32_t* C,
                        int64_t ldc, const DequantArgs* dq, tile::SmallPlan plan) {
  if (!any::tile_ok(M, N, K, 1, lda, ldb, !b_nk) || (dq && dq->acc_out)) return false;
  const bool split = b_nk ? launch_i8_layout<tile::B_NK>(ctx, M, N, K, A, lda, B, ldb, C, ldc, dq, plan)
                          : launch_i8_layout<tile::B_KN8>(ctx, M, N, K, A, lda, B, ldb, C, ldc, dq, plan);
  set_tile_kernel_name(ctx, "i8", 64,
                       dq ? (b_nk ? "_nk_dequant" : "_kn_dequant") : (b_nk ? "_nk" : "_kn"), split,
                       true);
  return true;
}

}  // namespace cig
