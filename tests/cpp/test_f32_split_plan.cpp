// Host-only check of the planner of the fp32 tiles on the bf16 matrix instructions
// (csrc/f32_split_plan.h): over a grid of sizes, K ranges are whole stages that the kernel takes, partial sums
// fit, columns are covered once, and no sum is longer than what the tile height may add up.
#include <cstdio>

#include "f32_split_plan.h"

using namespace cig;

static bool launch_ok(long long M, long long N, long long K, int rows, int wanted, long long length, size_t room) {
  int64_t range_k = 0;
  const int ranges = split32::k_ranges(K, wanted, &range_k);
  bool ok = rows >= 64 && rows <= 128 && rows % 32 == 0 && ranges >= 1 && ranges <= wanted &&
            range_k <= length + length / 4;
  if (ranges == 1) return ok && range_k == K;
  const long long last = K - (ranges - 1) * range_k;
  return ok && range_k % 16 == 0 && range_k >= 32 && last >= 17 && last <= range_k &&
         (size_t)ranges * M * ((N + 31) / 32 * 32) * 4 <= room;
}

// Every plan there is, one after the other; `est` as in split32::best_launch.
static split32::Plan each_launch(long long M, long long N, long long K, long long length, size_t room, double* est) {
  split32::Plan best{0, 1, 0, 0};
  for (int rows = 64; rows <= 128 && (rows == 64 || rows - 32 < M); rows += 32) {
    const long long tiles = (M + rows - 1) / rows * ((N + 255) / 256);
    for (int wanted = 1; wanted <= 32; ++wanted) {
      int64_t range_k = 0;
      const int sp = split32::k_ranges(K, wanted, &range_k);
      if (range_k > length + length / 4 ||
          (sp > 1 && (tiles * sp > 512 || range_k < 64 || (size_t)sp * M * ((N + 31) / 32 * 32) * 4 > room)))
        continue;
      const double us = split32::launch_us(M, N, K, 256, rows, sp);
      if (us < *est) *est = us, best = split32::Plan{rows, sp, 0, 0};
    }
  }
  return best;
}

static split32::Plan each(long long M, long long N, long long K, long long length, size_t room, double* est) {
  split32::Plan b = each_launch(M, N, K, length, room, est);
  for (int rows = 96; rows <= 128; rows += 32) {
    const long long tiles_m = (M + rows - 1) / rows, tiles_n = (N + 255) / 256;
    if (tiles_m > 256 || K > length + length / 4) continue;
    const long long cols = tiles_n / (256 / tiles_m) * (256 / tiles_m);
    if (cols <= 0 || cols >= tiles_n) continue;
    double us = 1e30;
    const double first = split32::launch_us(M, cols * 256, K, 256, rows, 1);
    const split32::Plan rest = each_launch(M, N - cols * 256, K, length, room, &us);
    if (rest.rows && first + us < *est) *est = first + us, b = split32::Plan{rest.rows, rest.ranges, cols * 256, rows};
  }
  return b;
}

int main() {
  for (long long K = 17; K < 3000; ++K)
    for (int wanted = 1; wanted <= 64; ++wanted)
      if (!launch_ok(1, 32, K, 64, wanted, 1LL << 40, (size_t)1 << 40)) {
        std::printf("FAILED K %lld wanted %d\n", K, wanted);
        return 1;
      }
  const long long Ms[] = {1, 33, 64, 65, 100, 257, 1000, 3000, 20000, 2000000};
  const long long Ns[] = {2, 16, 255, 256, 257, 1000, 4097, 16384};
  const long long Ks[] = {17, 32, 33, 784, 4099, 16384, 1000000};
  int plans = 0, pairs = 0, none = 0;
  for (long long M : Ms)
    for (long long N : Ns)
      for (long long K : Ks)
        for (long long length : {K, K / 4 + 1, 64LL})
          for (size_t room : {(size_t)0, (size_t)1 << 20, (size_t)64 << 20}) {
            double us = 1e30, each_us = 1e30;
            const split32::Plan p = split32::best(M, N, K, length, 256, room, &us);
            // nothing better is passed over, and nothing is found where all are above the limit
            const split32::Plan q = each(M, N, K, length, room, &each_us);
            double limit = 0.999999 * each_us, above = 1.3 * each_us;
            if (p.rows != q.rows || p.ranges != q.ranges || p.first_cols != q.first_cols ||
                p.first_rows != q.first_rows || us > each_us * 1.000001 ||
                (q.rows && (split32::best(M, N, K, length, 256, room, &limit).rows ||
                            split32::best(M, N, K, length, 256, room, &above).rows != p.rows))) {
              std::printf("FAILED %lld %lld %lld length %lld: %d x %d, of all plans %d x %d\n", M, N, K, length, p.rows,
                          p.ranges, q.rows, q.ranges);
              return 1;
            }
            bool ok = p.rows == 0 || (us > 0 && launch_ok(M, N - p.first_cols, K, p.rows, p.ranges, length, room));
            if (p.first_cols)
              ok = ok && p.first_cols % 256 == 0 && p.first_cols > 0 && p.first_cols < N &&
                   launch_ok(M, p.first_cols, K, p.first_rows, 1, length, room);
            // (with the whole K as the other kernel's sum one range always may)
            if (length == K) ok = ok && p.rows;
            if (!ok) {
              std::printf("FAILED %lld %lld %lld length %lld room %zu: rows %d ranges %d first %lld x %d\n", M, N, K,
                          length, room, p.rows, p.ranges, (long long)p.first_cols, p.first_rows);
              return 1;
            }
            ++(p.first_cols ? pairs : p.rows ? plans : none);
          }
  if (split32::ok(1, 1, 32, 32, 1) || split32::ok(1, 8, 16, 16, 8) || split32::ok(1, 8, 32, 1LL << 21, 8) ||
      split32::ok(1, 8, 32, 32, 1LL << 21) || !split32::ok(1, 2, 17, 17, 2)) {
    std::printf("FAILED ok\n");
    return 1;
  }
  std::printf("f32 split plan OK: %d plans, %d of two launches, %d without\n", plans, pairs, none);
  return plans > 300 && pairs > 10 && none > 5 ? 0 : 1;
}
