// fp32 GEMM and linear layer on the bf16 matrix instructions (f32_split_tile.h): launching a plan, and which
// calls of CIGEMM_ALGO_DEFAULT are taken.
#include "epilogues.h"
#include "f32_split_plan.h"
#include "kwaves_plan.h"
#include "mfma_tile.h"

namespace cig {
namespace split32 {
// (f32_split_rows.hip, once for each height)
template <int ROWS, typename Epi>
void launch(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, int64_t range_k, int ranges, const float* A,
            int64_t lda, const float* B, int64_t ldb, const Epi& epi);
}  // namespace split32

namespace {

template <typename Epi>
void launch_rows(cigemmContext* ctx, int rows, int64_t M, int64_t N, int64_t K, int64_t range_k, int ranges,
                 const float* A, int64_t lda, const float* B, int64_t ldb, const Epi& epi) {
#define CIG_ROWS(R) \
  case R: return split32::launch<R>(ctx, M, N, K, range_k, ranges, A, lda, B, ldb, epi)
  switch (rows) {
    CIG_ROWS(64); CIG_ROWS(96);
    default: return split32::launch<128>(ctx, M, N, K, range_k, ranges, A, lda, B, ldb, epi);
  }
#undef CIG_ROWS
}

// One launch, or one per K range and the reduction; true in the second case.
template <typename Epi>
bool run(cigemmContext* ctx, int rows, int wanted, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
         const float* B, int64_t ldb, const Epi& epi) {
  int64_t range_k = K;
  int ranges = split32::k_ranges(K, wanted, &range_k);
  const int64_t ld = tile::partial_ld<true>(N);
  if (ranges > 1 && (!ctx->workspace || (size_t)ranges * (size_t)M * (size_t)ld * 4 > ctx->ws_partial_bytes))
    ranges = split32::k_ranges(K, 1, &range_k);
  if (ranges == 1) {
    launch_rows(ctx, rows, M, N, K, range_k, 1, A, lda, B, ldb, epi);
    return false;
  }
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  uint32_t* ws = static_cast<uint32_t*>(ctx->workspace);
  launch_rows(ctx, rows, M, N, K, range_k, ranges, A, lda, B, ldb, tile::EpiPartialX4{ws, ld, M * ld});
  const int64_t blocks = any::div_up(M * any::div_up(N, 4), 256);
  hipLaunchKernelGGL((tile::splitk_reduce_kernel<float, Epi, true>),
                     dim3((unsigned)(blocks < 4 * (int64_t)cus ? blocks : 4 * (int64_t)cus)), dim3(256), 0,
                     ctx->stream, (int)M, (int)N, ranges, ws, M * ld, epi);
  return true;
}

template <typename Epi>
bool run_plan(cigemmContext* ctx, const split32::Plan& plan, int64_t M, int64_t N, int64_t K, const float* A,
              int64_t lda, const float* B, int64_t ldb, const Epi& epi) {
  const int64_t n1 = plan.first_cols;
  if (n1) run(ctx, plan.first_rows, 1, M, n1, K, A, lda, B, ldb, epi);
  const int rows1 = n1 ? ctx->last_tile_rows : 0;
  const bool split = run(ctx, plan.rows, plan.ranges, M, N - n1, K, A, lda, B + n1, ldb, epi.shift_cols(n1));
  ctx->first_tile_rows = rows1;
  ctx->first_waves = n1 ? 4 : 0;
  return split;
}

void launch_plan(cigemmContext* ctx, const split32::Plan& plan, bool any, int64_t M, int64_t N, int64_t K,
                 const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                 const BiasAct* ba) {
  const bool split =
      ba ? run_plan(ctx, plan, M, N, K, A, lda, B, ldb, EpiBiasActAnyF32x4{C, ldc, ba->bias, ba->relu})
         : run_plan(ctx, plan, M, N, K, A, lda, B, ldb, EpiStoreF32x4{C, ldc});
  const bool two = ctx->first_tile_rows != 0;
  char rows[32];
  if (two)
    snprintf(rows, sizeof(rows), "%d+%d", ctx->first_tile_rows, ctx->last_tile_rows);
  else
    snprintf(rows, sizeof(rows), "%d", ctx->last_tile_rows);
  snprintf(ctx->kernel_name, sizeof(ctx->kernel_name), "f32_mfma_%s%sx256x16_%s_ring4%s%s", any ? "any_" : "", rows,
           two ? "w4+w4" : "w4", ba ? "_bias_act" : "", split ? "_splitk" : "");
  ctx->last_kernel = ctx->kernel_name;
}

// What CIGEMM_ALGO_DEFAULT does with a call: `plan.rows` = 0 leaves it to the other kernels; `rest`: so many of the
// last columns by the kernel of small outputs, the others by the plan.
struct Choice {
  split32::Plan plan;
  int64_t rest;
};

// The two estimates err by 4 and 11 %: this one has to be 8 % below.  The small kernel's is up to 25 % too high for K
// of 500 to 1000 (1454 x 896 x 704 26.5 us there, 31.5 here): 16 %.  Of 6203 random calls taken with 8 % everywhere (M
// 65..20000, N 16..16384, K 17..16384, both kernels in turn) 40 were more than 3 % slower, 34 of them of
// the small kernel's 299; 6132 are taken with both, 1.16 times as fast (geometric mean), nine more than 3 % slower
// (the worst 6 %).
constexpr double MARGIN = 0.92, MARGIN_SMALL = 0.84;

Choice choose(const cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B,
              int64_t ldb, const float* C, int64_t ldc, const BiasAct* ba) {
  const Choice none{split32::Plan{0, 1, 0, 0}, 0};
  // A tile of up to 64 rows streams a long B more slowly than estimated (62 x 12032 x 7744 117 us, fp32
  // instructions 107).  Below 3e8 products the estimates took three of 1962 sizes, none of them
  // faster here, and they are host time.
  if (M <= 64 || (double)M * (double)N * (double)K < 3e8) return none;
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const size_t room = ctx->workspace ? ctx->ws_partial_bytes : 0;
  // the kernel that serves the call otherwise
  const F32Other other = f32_other(ctx, M, N, K, A, lda, B, ldb, C, ldc, ba);
  double us = 0;
  // (the kernel of small outputs' calls stay there: of its short sums only K in many ranges here is an equal,
  // and one of 900 such sizes was more than 3 % faster)
  if (any::tile_ok(M, N, K, 4, lda, ldb, true) && !(K <= 512 && f32_small_is_narrow(M, N, K, A, lda)) &&
      kwaves::best_f32(M, N, K, cus, room, ctx->ws_counter_bytes, &us).splits && us < other.us)
    return none;
  us = (other.small ? MARGIN_SMALL : MARGIN) * other.us;
  const split32::Plan plan = split32::best(M, N, K, other.sum_length, cus, room, &us);
  // Up to 64 columns beyond whole tiles: the kernel of small outputs (4095 x 4097 x 4099 838 us;
  // the 4097th column as tiles over 8 ranges of K would take 50).
  const int64_t rest = N % tile::BN, n1 = N - rest;
  if (rest && rest <= 64 && n1) {
    double rest_us = 0;
    if (kwaves::best_f32(M, rest, K, cus, room, ctx->ws_counter_bytes, &rest_us).splits) {
      us -= rest_us;
      const split32::Plan main = split32::best(M, n1, K, other.sum_length, cus, room, &us);
      if (main.rows) return Choice{main, rest};
    }
  }
  return Choice{plan, 0};
}

}  // namespace

bool launch_f32_split(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                      const float* B, int64_t ldb, float* C, int64_t ldc, const BiasAct* ba) {
  if (ctx->force_split_rows < 0 || !split32::ok(M, N, K, lda, ldb)) return false;
  const bool any = !f32_tile_ok(M, N, K, A, lda, B, ldb, C, ldc, ba);
  if (ctx->force_split_rows > 0) {
    launch_plan(ctx, split32::Plan{ctx->force_split_rows, ctx->force_split_ranges, 0, 0}, any, M, N, K, A, lda, B,
                ldb, C, ldc, ba);
    return true;
  }
  // (a plan of another kernel is imposed)
  if (ctx->force_tile_rows || ctx->force_kwaves) return false;
  const Choice c = choose(ctx, M, N, K, A, lda, B, ldb, C, ldc, ba);
  if (!c.plan.rows) return false;
  if (!c.rest) {
    launch_plan(ctx, c.plan, any, M, N, K, A, lda, B, ldb, C, ldc, ba);
    return true;
  }
  const int64_t n1 = N - c.rest;
  BiasAct shifted{};
  if (ba) shifted = BiasAct{ba->bias ? ba->bias + n1 : nullptr, ba->relu};
  if (!launch_kwaves_f32(ctx, M, c.rest, K, A, lda, B + n1, ldb, C + n1, ldc, ba ? &shifted : nullptr, true))
    return false;
  launch_plan(ctx, c.plan, any, M, n1, K, A, lda, B, ldb, C, ldc, ba);
  char first[sizeof(ctx->kernel_name)];
  snprintf(first, sizeof(first), "%s", ctx->last_kernel);
  name_rest_columns(ctx, first);
  return true;
}

}  // namespace cig
