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
  // What fp32's estimate is compared with has the tile kernel's own heights: 96 and 160 rows here, where
  // this kernel is the slower one (us: K, here, there).
  const struct { long long M, N, K; double here, there; } other[] = {
      {67, 5568, 3392, 41.5, 38.9}, {68, 5696, 4416, 50.0, 47.1}, {86, 6848, 5568, 76.2, 69.3},
      {94, 8704, 2240, 44.5, 41.5}, {74, 6528, 8320, 102.5, 91.7},
      // two row tiles and more over a long stream of B, and many tiles
      {36, 5016, 7040, 59.5, 44.5}, {47, 11228, 4608, 85.0, 66.8}, {48, 11328, 3904, 72.9, 59.4},
      {54, 9920, 2496, 42.6, 35.4}, {104, 2048, 10176, 61.0, 47.6}, {467, 768, 7936, 64.4, 56.1},
      {420, 704, 7616, 56.2, 46.1}};
  const size_t room = (size_t)64 << 20;
  for (const auto& o : other) {
    double est = 0;
    kwaves::best_f32(o.M, o.N, o.K, 256, room, 65536, &est);
    const any::Problem p{o.M, o.N, 4 * o.K, 4, 4, false, false, false};
    const double there = any::other_us(any::COST_F32, p, true, 256, room);
    if (est <= there)
      return std::printf("FAILED fp32 %lld %lld %lld: %.1f here, %.1f there\n", o.M, o.N, o.K, est, there), 1;
  }
  // while these stay here
  const struct { long long M, N, K; double here, there; } kept[] = {
      {42, 6144, 2816, 22.9, 26.4}, {1, 5120, 7472, 39.1, 44.6}, {17, 9216, 3776, 38.5, 40.5}, {95, 896, 1344, 7.8, 17.1},
      {1995, 352, 12280, 185.1, 206.3}, {1708, 344, 13816, 191.2, 204.6}};  // (the long stream is A)
  for (const auto& o : kept) {
    double est = 0;
    kwaves::best_f32(o.M, o.N, o.K, 256, room, 65536, &est);
    const any::Problem p{o.M, o.N, 4 * o.K, 4, 4, false, false, false};
    const double there = any::other_us(any::COST_F32, p, true, 256, room);
    if (est >= there)
      return std::printf("FAILED fp32 %lld %lld %lld: %.1f here, %.1f there\n", o.M, o.N, o.K, est, there), 1;
  }
  // and its times: one round of 160-row tiles (130 us), three of 160 rows (420)
  const struct { long long M, N, K; double us; } times[] = {{20000, 512, 784, 130}, {3000, 3000, 3000, 420}};
  for (const auto& o : times) {
    const any::Problem p{o.M, o.N, 4 * o.K, 4, 4, false, false, false};
    const double us = any::other_us(any::COST_F32, p, true, 256, room);
    if (us < 0.93 * o.us || us > 1.07 * o.us)
      return std::printf("FAILED fp32 %lld %lld %lld: %.1f us\n", o.M, o.N, o.K, us), 1;
  }
  // 16-bit and int8: long streams of k that the tile kernel is the faster for, and some that stay here
  const struct { int elem; bool nk; long long M, N, K; double here, there; } streams[] = {
      {1, true, 787, 392, 15048, 29.8, 22.1}, {1, true, 8672, 128, 6088, 36.2, 27.6},
      {1, true, 2234, 144, 12464, 25.4, 19.4}, {2, false, 904, 276, 3896, 17.6, 14.1},
      {2, false, 1337, 232, 3944, 17.9, 15.0}, {2, false, 757, 570, 3856, 18.3, 15.9},
      {1, false, 77, 3112, 5408, 16.3, 14.0},
      {2, false, 50, 7648, 3264, 12.5, 16.0}, {2, false, 112, 3776, 2888, 11.6, 14.0}, {1, true, 285, 4384, 3200, 14.2, 18.7},
      {1, true, 61, 9352, 4096, 12.4, 15.6}};
  for (const auto& o : streams) {
    const any::Problem p{o.M, o.N, o.K * o.elem, o.elem, o.elem == 2 ? 2 : 4, false, false, false};
    const bool whole = p.K_bytes % 128 == 0 && (o.nk || o.N * o.elem % 16 == 0);
    const bool aligned = p.K_bytes % 16 == 0 && o.N * (o.nk ? p.out_bytes : o.elem) % 16 == 0;
    const kwaves::Cost& c =
        o.elem == 2 ? kwaves::COST_16 : o.nk ? kwaves::COST_I8_NK : kwaves::COST_I8_KN;
    const any::Cost& other = o.elem == 2 ? any::COST_16 : o.nk ? any::COST_I8_NK : any::COST_I8_KN;
    const bool taken_here = kwaves::choose(c, other, p, whole, aligned, 256, room, 65536).splits > 0;
    if (taken_here != (o.here < o.there))
      return std::printf("FAILED %lld x %lld x %lld: %.1f us here, %.1f there\n", o.M, o.N, o.K, o.here, o.there), 1;
  }
  if (taken < 100 || refused < 100) return std::printf("FAILED: %d taken, %d refused\n", taken, refused), 1;
  std::printf("kwaves plan OK\n");
  return 0;
}
