// The fp32 tiles on the bf16 matrix instructions of one height (CIG_SPLIT_ROWS, given on the compiler's
// command line: a file each, since a kernel takes ten seconds to compile).
#include "epilogues.h"
#include "f32_split_tile.h"

namespace cig {
namespace split32 {

template <int ROWS, typename Epi>
void launch(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, int64_t range_k, int ranges, const float* A,
            int64_t lda, const float* B, int64_t ldb, const Epi& epi) {
  typedef tile::SplitTile<ROWS / 32> S;
  static_assert(S::TILE_M == ROWS, "");
  auto kern = tile::f32_split_kernel<ROWS / 32, Epi>;
  static std::atomic<uint64_t> lds_set{0};
  if (!ensure_dynamic_lds(ctx, (const void*)kern, S::LDS_BYTES, lds_set)) return;
  const int tiles_m = (int)((M + ROWS - 1) / ROWS), tiles_n = (int)((N + tile::BN - 1) / tile::BN);
  ctx->last_tile_rows = ROWS;
  ctx->last_k_splits = ranges;
  ctx->last_waves = 4;
  ctx->last_per_cu = 1;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n), (unsigned)ranges), dim3(256), S::LDS_BYTES,
                     ctx->stream, (int)M, (int)N, (int)K, (int)range_k, tiles_m, tiles_n, A, lda, B, ldb, epi);
}

#define CIG_INSTANCE(Epi)                                                                                  \
  template void launch<CIG_SPLIT_ROWS, Epi>(cigemmContext*, int64_t, int64_t, int64_t, int64_t, int, const float*, \
                                            int64_t, const float*, int64_t, const Epi&)
CIG_INSTANCE(EpiStoreF32x4);
CIG_INSTANCE(EpiBiasActAnyF32x4);
CIG_INSTANCE(tile::EpiPartialX4);

}  // namespace split32
}  // namespace cig
