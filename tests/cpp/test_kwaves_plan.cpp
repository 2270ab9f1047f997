// Host-only check of the planner of the kernel of small outputs (csrc/kwaves_plan.h): over a grid of
// sizes, what it plans fits the launch, the partial sums, the arrival counters and K, and it leaves the
// calls alone that the rules in front of its estimate name.
#include <cstdio>

#include "kwaves_plan.h"

using namespace cig;

int main() {
  const long long Ms[] = {1, 17, 32, 33, 100, 300, 1000, 3000, 40000};
  const long long Ns[] = {8, 15, 16, 64, 65, 1000, 4096, 16384};
  const long long Ks[] = {16, 384, 385, 1000, 2048, 8192, 65536, 2147483647LL};
  int taken = 0, refused = 0;
  for (long long M : Ms)
    for (long long N : Ns)
      for (long long K : Ks)
        for (size_t room : {(size_t)0, (size_t)1 << 20, (size_t)64 << 20})
          for (int aligned = 0; aligned < 2; ++aligned) {
            const any::Problem p{M, N, K, 1, 4, true, !aligned, !aligned};
            const size_t counters = 4096;
            const kwaves::Plan plan = kwaves::choose(kwaves::COST_I8_KN, any::COST_I8_KN, p, aligned,
                                                     aligned, 256, room, counters);
            const long long tiles = any::div_up(M, 32) * any::div_up(N, 64);
            const bool never = K <= 384 || N < 16 || tiles > 768;
            int64_t stages = 0;
            const int ranges = tile::k_ranges(K, plan.splits, &stages);
            bool ok = plan.splits >= 0 && plan.splits <= 16 && !(never && plan.splits);
            if (plan.splits > 1)
              ok = ok && ranges >= 1 && stages % 2 == 0 && (ranges - 1) * stages * 64 < K &&
                   tiles * plan.splits * 8192 <= (long long)room && tiles * 4 <= (long long)counters;
            if (!ok) {
              std::printf("FAILED %lld %lld %lld room %zu: %d ranges\n", M, N, K, room, plan.splits);
              return 1;
            }
            ++(plan.splits ? taken : refused);
          }
  // fp32: the same, no range longer than 8 KiB of k
  for (long long M : Ms)
    for (long long N : Ns)
      for (long long K : {16LL, 64LL, 65LL, 1000LL, 2048LL, 2049LL, 30000LL, 40000LL, 500000000LL})
        for (size_t room : {(size_t)0, (size_t)1 << 20, (size_t)64 << 20}) {
          double est = 0;
          const size_t counters = 4096;
          const kwaves::Plan plan = kwaves::best_f32(M, N, K, 256, room, counters, &est);
          const long long tiles = any::div_up(M, 32) * any::div_up(N, 32);
          int64_t stages = 0;
          const int ranges = tile::k_ranges(4 * K, plan.splits, &stages);
          bool ok = !((K <= 64 || tiles > 1024 || K > 32768) && plan.splits) && plan.splits <= 16;
          if (plan.splits) ok = ok && est > 4.0 && est < 1e6 && stages * 64 <= 8192 + 128;
          if (plan.splits > 1)
            ok = ok && stages % 2 == 0 && (ranges - 1) * stages * 64 < 4 * K &&
                 tiles * plan.splits * 4096 <= (long long)room && tiles * 4 <= (long long)counters;
          if (!ok) {
            std::printf("FAILED fp32 %lld %lld %lld room %zu: %d ranges\n", M, N, K, room, plan.splits);
            return 1;
          }
          ++(plan.splits ? taken : refused);
        }
  if (taken < 100 || refused < 100) return std::printf("FAILED: %d taken, %d refused\n", taken, refused), 1;
  std::printf("kwaves plan OK\n");
  return 0;
}
