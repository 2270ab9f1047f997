// Host-only check of the choice among the any-alignment kernels (csrc/any_plan.h).  Reads lines
//   kind M N K out_bytes dequant narrow
// (kind: bf16, f32, i8kn, i8nk; K in elements; packed matrices; narrow: the small fp32 kernel runs its
// 16 x 16 form) and prints the estimates "tile staged small" in us, -1 where a kernel does not take
// the call, as the library has them on 256 compute units with 64 MiB of partial sums.
#include <cstdio>
#include <cstring>

#include "any_plan.h"

using namespace cig;

int main() {
  char kind[16];
  long long M, N, K;
  int out_bytes, dequant, narrow;
  const size_t room = (size_t)64 << 20;
  while (std::scanf("%15s %lld %lld %lld %d %d %d", kind, &M, &N, &K, &out_bytes, &dequant, &narrow) == 7) {
    const bool f32 = !std::strcmp(kind, "f32"), nk = !std::strcmp(kind, "i8nk");
    const int elem = f32 ? 4 : !std::strcmp(kind, "bf16") ? 2 : 1;
    const any::Cost& c = f32 ? any::COST_F32 : elem == 2 ? any::COST_16 : nk ? any::COST_I8_NK : any::COST_I8_KN;
    const long long ldb = nk ? K : N;
    const any::Problem p{M, N, K * elem, elem, out_bytes, dequant != 0, (K * elem & 3) != 0, (ldb * elem & 3) != 0};
    int64_t steps = 0;
    const int sp = any::staged_ranges(p, 256, room, &steps);
    const int64_t all = any::div_up(p.K_bytes, 64);
    // the ranges cover K, none is empty, the partial sums fit
    if (sp < 1 || sp > 16 || sp * steps < all || (sp - 1) * steps >= all ||
        (sp > 1 && (size_t)sp * M * N * 4 > room)) {
      std::printf("FAILED %s %lld %lld %lld: %d ranges of %lld steps\n", kind, M, N, K, sp, (long long)steps);
      return 1;
    }
    const bool tile = any::tile_ok(M, N, K, elem, K, ldb, !nk);
    std::printf("%.4f %.4f %.4f\n", tile ? any::tile_us(c, p, 256, room, any::tile_plan(c, p, 256, room)) : -1.0,
                any::staged_us(c, p, 256, room),
                f32 ? any::f32_small_us(M, N, K, 256, N % 4 == 0, narrow != 0) : -1.0);
  }
  return 0;
}
