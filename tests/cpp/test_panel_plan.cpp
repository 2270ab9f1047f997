// Host-only check of which calls the kernel of batches (csrc/panel_plan.h) takes: none that was slower there by
// more than the estimates err, those that it is for, and no more tiles than one round.
#include <cstdio>

#include "panel_plan.h"

using namespace cig;

static int rows_of(bool int8, long long M, long long N, long long K, int out_bytes, bool dequant) {
  const any::Problem p{M, N, int8 ? K : 2 * K, int8 ? 1 : 2, out_bytes, dequant, false, false};
  return panel::choose(int8 ? panel::COST_I8_NK : panel::COST_16, int8 ? any::COST_I8_NK : any::COST_16, p, 256,
                       (size_t)64 << 20);
}

struct Call {
  bool int8;
  long long M, N, K;
  int out_bytes;
};

int main() {
  // us, tile kernel and here
  const Call slower[] = {{false, 67, 13936, 2544, 2},   // 23.9, 27.2
                         {false, 1860, 720, 2768, 2},   // 21.3, 24.5
                         {false, 1915, 640, 2608, 2},   // 19.8, 21.4
                         {true, 216, 6464, 13328, 2},   // 54.3, 71.1
                         {true, 223, 6480, 14960, 4},   // 60.1, 72.7
                         {true, 1378, 784, 5104, 2},    // 22.5, 25.7
                         {true, 354, 2816, 5840, 2}};   // 22.0, 24.7
  const Call faster[] = {{false, 229, 2752, 1984, 2},   // 17.4, 11.9
                         {false, 1097, 1664, 1664, 2},  // 19.0, 13.6
                         {true, 256, 4096, 4096, 2},    // 17.3, 12.7
                         {true, 512, 4096, 4096, 2}};   // 22.8, 17.0
  for (const Call& c : slower)
    if (rows_of(c.int8, c.M, c.N, c.K, c.out_bytes, c.int8 && c.out_bytes == 2)) {
      std::printf("FAILED taken: %lld %lld %lld\n", c.M, c.N, c.K);
      return 1;
    }
  for (const Call& c : faster)
    if (!rows_of(c.int8, c.M, c.N, c.K, c.out_bytes, c.int8 && c.out_bytes == 2)) {
      std::printf("FAILED not taken: %lld %lld %lld\n", c.M, c.N, c.K);
      return 1;
    }
  int taken = 0;
  for (long long M = 1; M < 3000; M += 37)
    for (long long N = 16; N < 20000; N += 16 + N / 8 / 16 * 16)
      for (long long K = 64; K < 20000; K += 64 + K / 8 / 64 * 64)
        for (bool int8 : {false, true})
          if (const int rows = rows_of(int8, M, N, K, 2, int8)) {
            ++taken;
            if ((rows != 64 && rows != 128) || any::div_up(M, rows) * any::div_up(N, panel::TN) > 256 || M <= 32) {
              std::printf("FAILED %lld %lld %lld: %d rows\n", M, N, K, rows);
              return 1;
            }
          }
  std::printf("panel plan OK: %d taken\n", taken);
  return taken > 1000 ? 0 : 1;
}
