// fp32 GEMM tiles on the bf16 matrix instructions, every operand held exactly.
//
// An fp32 number of 24 bits is the sum of three bf16 numbers of 8: h = bf16(x), m = bf16(x - h), l = x - h -
// m, every difference exact.  a b is then h h' + (h m' + m h') + (m m' + h l' + l h') + (m l' + l m') and l l', below
// 2^-32 of it, which is left out: eight v_mfma_f32_32x32x16_bf16 in place of eight v_mfma_f32_32x32x2_f32
// for 16 of k, 256 cycles in place of 512, sums in fp32 as before.
// h h' has a running sum of its own, the seven smaller products another, and the two meet at the end: a rounding of
// the large sum for eight of k, where the fp32 instruction rounds for each one.  Error against 64 bits, by the
// fp32 instructions' on the same operands (131072 outputs each, K = 64, 1024 and 4096): 0.30 to 0.33 for dense
// operands, 0.32 to 0.83 for rows with 2 nonzero values up to 60 % of them, and where one product makes the result
// the same to four digits (at most 0.51 units in the last place, 0.50 there).  With one running sum that ratio is 0.75 to
// 0.87 for dense operands but up to 2.0 for sparse ones (each of the products rounds the sum, where the fp32
// instruction adds zeros), and without m l' + l m' a lone product is off by up to 0.91 units: neither is kept,
// though tiles of 256 rows, whose registers hold one sum only, take 743 us for 4096^3, and six products 668 here.
// The host takes the tiles only where no sum gets longer by more than the rest allows (f32_split_plan.h,
// range_limit).
//
// What three parts cannot hold: infinities and NaN (x - h is NaN), magnitudes that bf16 rounds to infinity,
// and below 2^-110, where the last part falls short of bf16's subnormals: there up to 2^-134 of the value is lost, and
// of a result K 2^-133 times the largest magnitude of the tile's operands.  A workgroup that got a result that is not
// finite, or met such small values and got a result of which that would be more than 2^-34, computes its tile
// once more with the fp32 instructions, straight from memory, on top of the first pass.  (So a small value among
// ordinary ones, the tail of a softmax or a decayed weight, changes nothing, unless a row or column of the
// tile gives zero or next to it.)  us, 4096^3 with a value in every
// 64th row: 1e-35 813 (809 without; every tile again 2283), NaN 2014 (fp32 instructions 905).
//
// Workgroup = 256 lanes = 4 waves, tile of 64, 96 or 128 rows x 256 columns, stages of 16 k.  Values go from
// memory to registers (8 k of one row of A; 8 k of two columns of B, so that the matrix instruction's
// order of B needs no transposing read), are split there, once per workgroup, and written to LDS as the three parts in fragment
// order ([32 rows][16 k] blocks of 1 KiB, a lane's 16 bytes in one read, rows permuted so that reads and
// writes meet no bank conflict).  Any alignment: nothing here needs more than the elements'.
// One barrier a stage, behind the first matrix instructions; the parts of stage s + 2 are written under the
// multiplies of stage s, whose own fragments were read in the stage before; loads are two stages ahead of the
// splitting.  The order of the slots (one matrix instruction, its share of the splitting, at most a read, a write and a
// load) is pinned.
//
// What bounds it: the chip's power.  A tile takes the same cycles with one workgroup and with all units at work (75 % of
// them matrix instructions), but the clock falls from 2.49 to 1.81 GHz, and does not where the operands are zeros:
// 128 rows 1120 ns a stage with one workgroup, 1565 with 256, 1132 with 256 on zeros (profiles/fp32_bf16_parts.md).
// fp32 instructions -> here, one process, us: 4096^3 905 -> 809, 4095 x 4097 x 4099 930 -> 838, 256 x 8192 x 8192 244 -> 226.
#pragma once

#include "mfma_tile.h"

namespace cig {
namespace tile {

// f(0), f(1) .. f(n - 1), each with its number as a constant
template <typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// MT x NT blocks of 32 x 32 a wave, the waves side by side.
template <int MT>
struct SplitTile {
  static constexpr int NT = BN / 4 / 32;
  static constexpr int TILE_M = 32 * MT;
  static_assert(MT >= 2 && MT <= 4, "two sums of a block fill the accumulator registers at 128 rows");
  static constexpr int KS = 16;                       // k of a stage: one matrix instruction's
  static constexpr int A_BLOCKS = 4, B_BLOCKS = 8;    // (A's are fetched and split as of 128 rows)
  static constexpr int BLOCK = 1024;                  // 32 rows (columns) x 16 k of one part
  static constexpr int A_BYTES = 3 * A_BLOCKS * BLOCK, SLOT = A_BYTES + 3 * B_BLOCKS * BLOCK;
  static constexpr int RING = 4;
  static constexpr int LDS_BYTES = RING * SLOT + 16;
  static constexpr int PRODUCTS = 8;
  static constexpr int MFMAS = PRODUCTS * MT * NT;    // per stage and wave
  static constexpr int TASKS = 3;                     // groups of 8 elements a lane splits per stage: B, B, A
};

// The running sums of an output block.
struct MathSplit {
  struct acc_t {
    f32x16 part[2];  // of h h' and of the smaller products
    __device__ __forceinline__ float operator[](int e) const { return part[0][e]; }
  };
};
// An epilogue that also notes whether any value was infinite or not a number, and the smallest magnitude.
template <typename Epi>
struct EpiChecked : Epi {
  float &check, &smallest;
  __device__ __forceinline__ EpiChecked(const Epi& e, float& c, float& s) : Epi(e), check(c), smallest(s) {}
  template <typename R, typename C>
  __device__ __forceinline__ u32x4 pack(R r, C c, float v0, float v1, float v2, float v3) const {
    check = __builtin_fmaf(v0, 0.0f, check);
    check = __builtin_fmaf(v1, 0.0f, check);
    check = __builtin_fmaf(v2, 0.0f, check);
    check = __builtin_fmaf(v3, 0.0f, check);
    smallest = __builtin_fminf(__builtin_fminf(smallest, __builtin_fabsf(v0)), __builtin_fabsf(v1));
    smallest = __builtin_fminf(__builtin_fminf(smallest, __builtin_fabsf(v2)), __builtin_fabsf(v3));
    return Epi::pack(r, c, v0, v1, v2, v3);
  }
};

template <int MT, typename Epi>
__global__ __launch_bounds__(256, 1) void f32_split_kernel(int M, int N, int K_total, int range_k,
                                                           int tiles_m, int tiles_n,
                                                           const float* __restrict__ A, int64_t lda,
                                                           const float* __restrict__ B, int64_t ldb,
                                                           Epi epi_all) {
  // blockIdx.y = K range
  const int k_from = (int)blockIdx.y * range_k;
  const int K = K_total - k_from < range_k ? K_total - k_from : range_k;
  A += k_from;
  B += (int64_t)k_from * ldb;
  const Epi epi = epilogue_of_split(epi_all, (int)blockIdx.y);
  typedef SplitTile<MT> S;
  constexpr int NT = S::NT;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int t = threadIdx.x, l = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  // the workgroup's: results not finite, values below 2^-110 met, largest operand, smallest result (bits)
  uint32_t* const vote = reinterpret_cast<uint32_t*>(lds + S::RING * S::SLOT);
  if (t < 4) vote[t] = t < 3 ? 0 : 0x7f800000;
  int tm, tn;
  tile_of_workgroup(tiles_m, tiles_n, tm, tn);
  tm = __builtin_amdgcn_readfirstlane(tm);
  tn = __builtin_amdgcn_readfirstlane(tn);
  const int64_t m0 = (int64_t)tm * S::TILE_M, n0 = (int64_t)tn * BN;

  // ---- what a lane fetches and splits --------------------------------------------------------
  // A: 8 k of a row.  B: 8 k of two columns (a wave 8 rows of k x 128 columns).  The last 1..16 of k
  // come first, element by element.
  const int full = (K - 1) / S::KS, tail = K - full * S::KS;
  // (the tail, and one of zeros where their number is odd: two stages a trip of the main loop)
  const int first = full % 2 == 0 ? 2 : 1;
  const int stages = full + first;
  const int a_half = t & 1, a_row = t >> 1;
  const int b_half = w & 1, b_col = 128 * (w >> 1) + 2 * l;
  const int b_left = N - n0 < BN ? (int)(N - n0) : BN;  // columns of the tile
  const int b_back = b_left == 1 ? 1 : 0;
  uint32_t a_voff, b_voff[8];
  {
    // (rows past the tile's re-read its last one)
    const int64_t last = M - m0 < S::TILE_M ? M - m0 - 1 : S::TILE_M - 1;
    a_voff = (uint32_t)((a_row < last ? a_row : last) * lda * 4) + a_half * 32;
    // (columns past N - 2 fetch the last two: what no row holds is read nowhere)
    const int64_t c = b_col < b_left - 2 ? b_col : b_left - 2;
#pragma unroll
    for (int j = 0; j < 8; ++j) b_voff[j] = (uint32_t)((c + b_back) * 4 + j * ldb * 4);
  }
  const char* const a_tile = reinterpret_cast<const char*>(A + m0 * lda);
  const char* const b_tile = reinterpret_cast<const char*>(B + n0 - b_back);
  // Whole stages are fetched one after the other; past the last one that one again, into slots nobody reads.
  const int64_t b_step = 16 * ldb * 4;
  const char *a_next = a_tile, *b_next = b_tile + b_half * (b_step / 2);
  int to_load = full;
  auto advance = [&]() {
    to_load -= 1;
    a_next += to_load > 0 ? 64 : 0;
    b_next += to_load > 0 ? b_step : 0;
  };
  typedef float raw_t[S::TASKS][8];
  raw_t raw[2];
  // (a lane offset the compiler may not widen outside the loop: scalar base + 32 bits is one instruction)
  auto load_b = [&](raw_t& x, int j) {
    uint32_t v = b_voff[j];
    asm volatile("" : "+v"(v));
    f32x2 q;
    __builtin_memcpy(&q, b_next + v, 8);
    x[0][j] = q[0];
    x[1][j] = q[1];
  };
  auto load_a = [&](raw_t& x, int half) {
    uint32_t v = a_voff;
    asm volatile("" : "+v"(v));
    f32x4 q;
    __builtin_memcpy(&q, a_next + v + 16 * half, 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[2][4 * half + e] = q[e];
  };
  auto load_stage = [&](raw_t& x) {
#pragma unroll
    for (int j = 0; j < 8; ++j) load_b(x, j);
#pragma unroll
    for (int q = 0; q < 2; ++q) load_a(x, q);
    advance();
  };
  auto load_tail = [&](raw_t& x, int valid) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int ka = a_half * 8 + j, kb = b_half * 8 + j;
      const float a = *reinterpret_cast<const float*>(a_tile + (a_voff - a_half * 32) +
                                                      (int64_t)(ka < valid ? full * 16 + ka : K - 1) * 4);
      x[2][j] = ka < valid ? a : 0.0f;
      const float* row = reinterpret_cast<const float*>(
          b_tile + (int64_t)(kb < valid ? full * 16 + kb : K - 1) * ldb * 4 + b_voff[0]);
      const float b0 = row[0], b1 = row[1];
      x[0][j] = kb < valid ? b0 : 0.0f;
      x[1][j] = kb < valid ? b1 : 0.0f;
    }
  };

  // ---- splitting -----------------------------------------------------------------------------
  const int r32 = l & 31;
  const uint32_t rd_a = (l >> 5) * 512 + ((r32 ^ ((l >> 5) << 2)) << 4);
  const uint32_t rd_b =
      S::A_BYTES + w * NT * S::BLOCK + (l >> 5) * 512 + (((r32 >> 1) ^ (r32 & 1 ? 20 : 0)) << 4);
  const uint32_t wr_a = (a_row >> 5) * S::BLOCK + a_half * 512 + (((a_row & 31) ^ (a_half << 2)) << 4);
  uint32_t wr_b[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
    wr_b[c] = S::A_BYTES + (b_col >> 5) * S::BLOCK + b_half * 512 + (((l & 15) ^ (c ? 20 : 0)) << 4);
  // (an odd last column is the second of the lane's pair; the first goes where nothing is stored from)
  if (b_col == b_left - 1) {
    const uint32_t even = wr_b[0];
    wr_b[0] = wr_b[1];
    wr_b[1] = even;
  }
  uint32_t least = 0xffffffffu;
  float most = 0.0f;
  auto part_of = [&](const float (&x)[8], int i) { return f32x2_to_bf16_bits(x[2 * i], x[2 * i + 1]); };
  auto rest_of = [&](float (&x)[8], uint32_t h, int i) {
    x[2 * i] -= __builtin_bit_cast(float, h << 16);
    x[2 * i + 1] -= __builtin_bit_cast(float, h & 0xffff0000u);
  };
  // smallest nonzero magnitude (twice its bits less one: zero comes out largest) and largest one
  auto watch = [&](const float (&x)[8], int i) {
    uint32_t u, v;
    asm volatile("v_lshl_add_u32 %2, %4, 1, -1\n\tv_lshl_add_u32 %3, %5, 1, -1\n\tv_min3_u32 %0, %0, %2, %3\n\t"
                 "v_max3_f32 %1, %1, |%4|, |%5|"
                 : "+v"(least), "+v"(most), "=&v"(u), "=&v"(v)
                 : "v"(x[2 * i]), "v"(x[2 * i + 1]));
  };
  auto put = [&](uint32_t slot, int task, int plane, u32x4 v) {
    const uint32_t at = task < 2 ? wr_b[task] + plane * S::B_BLOCKS * S::BLOCK
                                 : wr_a + plane * S::A_BLOCKS * S::BLOCK;
    *reinterpret_cast<u32x4*>(lds + slot + at) = v;
  };
  u32x4 part;
  // step d (0..11) of splitting task q
  auto split_step = [&](raw_t& x, uint32_t slot, int q, int d) {
    if (d < 2 || d == 6 || d == 11) {
      const int from = d < 2 ? 2 * d : 0, upto = d < 2 ? from + 2 : 4;
#pragma unroll
      for (int i = from; i < upto; ++i) {
        const uint32_t h = part_of(x[q], i);
        part[i] = h;
        if (d < 2) watch(x[q], i);
      }
    } else {
      const int i = d < 6 ? d - 2 : d - 7;
      const uint32_t h = part[i];
      rest_of(x[q], h, i);
    }
    if (d == 5 || d == 10 || d == 11) put(slot, q, d == 5 ? 0 : d == 10 ? 1 : 2, part);
  };
  auto split_stage = [&](raw_t& x, uint32_t slot) {
#pragma unroll
    for (int q = 0; q < S::TASKS; ++q)
#pragma unroll
      for (int d = 0; d < 12; ++d) split_step(x, slot, q, d);
  };
  auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // ---- prologue ------------------------------------------------------------------------------
  load_tail(raw[0], tail);
  if (first > 1) load_tail(raw[1], 0); else load_stage(raw[1]);
  split_stage(raw[0], 0);
  load_stage(raw[0]);
  split_stage(raw[1], S::SLOT);
  load_stage(raw[1]);
  barrier();

  MathSplit::acc_t acc[MT][NT];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j].part[c][e] = 0.0f;

  u32x4 fa[2][3], fb[3][NT];
  auto read_a = [&](uint32_t slot, int pl, int i) {
    return *reinterpret_cast<const u32x4*>(lds + slot + rd_a + (pl * S::A_BLOCKS + i) * S::BLOCK);
  };
  auto read_b = [&](uint32_t slot, int pl, int j) {
    return *reinterpret_cast<const u32x4*>(lds + slot + rd_b + (pl * S::B_BLOCKS + j) * S::BLOCK);
  };
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
    for (int j = 0; j < NT; ++j) fb[pl][j] = read_b(0, pl, j);
    fa[0][pl] = read_a(0, pl, 0);
  }

  // One stage: MFMAS slots of one matrix instruction and a handful of others.  `now` is multiplied,
  // `next` the stage after it, `to` the one after that, which the splitting fills.
  auto stage = [&](uint32_t now, uint32_t next, uint32_t to, auto u_) {
    constexpr int CUR = decltype(u_)::value, P = S::PRODUCTS;
    constexpr int STEPS = 12 * S::TASKS, SPLIT_SLOTS = S::MFMAS - 2, BARRIER_SLOT = 1;
    // (nothing is written before the barrier behind which every wave is done with the stage before)
    static_assert(5 * SPLIT_SLOTS / STEPS > BARRIER_SLOT, "");
    // part products, h h' last: (a part, b part).  The B fragments of the next stage replace
    // this one's in the last row block, each part behind its last use.
    constexpr int PB[P] = {2, 2, 1, 1, 1, 0, 0, 0}, PA[P] = {1, 0, 2, 1, 0, 2, 1, 0};
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(acc[i][j].part[c]));
    each_of([&](auto slot_) {
      constexpr int slot = decltype(slot_)::value;
      constexpr int i = slot / (P * NT), in_row = slot % (P * NT), p = in_row / NT, j = in_row % NT;
      constexpr int fi = (i + CUR * MT) & 1;
      f32x16& c = acc[i][j].part[p < P - 1 ? 1 : 0];
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fb[PB[p]][j]),
                                                  __builtin_bit_cast(bf16x8, fa[fi][PA[p]]), c, 0, 0, 0);
      // fragments of the next row block, or of the next stage's first
      if constexpr (in_row == 3 || in_row == 5 || in_row == 7) {
        constexpr int pl = (in_row - 3) / 2;
        fa[fi ^ 1][pl] = i + 1 < MT ? read_a(now, pl, i + 1) : read_a(next, pl, 0);
      }
      if constexpr (i == MT - 1 && (p == 1 || p == 4 || p == 7)) {
        constexpr int pl = p == 1 ? 2 : p == 4 ? 1 : 0;
        fb[pl][j] = read_b(next, pl, j);
      }
      each_of([&](auto step_) {
        constexpr int step = decltype(step_)::value;
        if constexpr (step * SPLIT_SLOTS / STEPS == slot) split_step(raw[CUR], to, step / 12, step % 12);
      }, std::make_integer_sequence<int, STEPS>{});
      // the raw values of a later stage, into the registers the tasks have left
      constexpr int B_FROM = 24 * SPLIT_SLOTS / STEPS + 1, B_SPAN = 11 * SPLIT_SLOTS / STEPS;
      each_of([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        if constexpr (slot == B_FROM + k * B_SPAN / 8) load_b(raw[CUR], k);
      }, std::make_integer_sequence<int, 8>{});
      constexpr int A_FROM = (12 * S::TASKS * SPLIT_SLOTS - 1) / STEPS + 1;
      if constexpr (slot == A_FROM) load_a(raw[CUR], 0);
      if constexpr (slot == A_FROM + 1) load_a(raw[CUR], 1);
      if constexpr (slot == S::MFMAS - 1) advance();
      if constexpr (slot == BARRIER_SLOT) barrier();
      __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, S::MFMAS>{});
  };
  // Stage s lies in slot s % RING.
  uint32_t slot0 = 0, slot1 = S::SLOT, slot2 = 2 * S::SLOT, slot3 = (S::RING - 1) * S::SLOT;
  int s = 0;
  do {
    stage(slot0, slot1, slot2, std::integral_constant<int, 0>{});
    stage(slot1, slot2, slot3, std::integral_constant<int, 1>{});
    const uint32_t was0 = slot0, was1 = slot1;
    slot0 = slot2;
    slot1 = slot3;
    slot2 = was0;
    slot3 = was1;
    s += 2;
  } while (s < stages);

  // ---- results -------------------------------------------------------------------------------
  // (one block at a time, kept where the matrix instructions left it: all of them in vector registers
  // at once would not fit)
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      acc[i][j].part[0] += acc[i][j].part[1];
      asm volatile("" : "+a"(acc[i][j].part[0]));
      __builtin_amdgcn_sched_barrier(0);
    }
  float check = 0.0f;  // NaN once a result was not finite
  float smallest = __builtin_inff();
  __syncthreads();     // (every wave is past its last fragment read: store_tile uses the ring)
  store_tile<MathSplit, MT, 4, S::TILE_M, true, NT>(EpiChecked<Epi>{epi, check, smallest}, acc, lds, w, 0, w, m0, n0,
                                                    M, N, 0.0f, 0.0f);
  // ---- what the split cannot hold: the tile once more, in fp32 ---------------------------------
  if (check != 0.0f) vote[0] = 1;
  if (least < (17u << 24) - 1) vote[1] = 1;
  __syncthreads();
  if (!__builtin_amdgcn_readfirstlane(vote[0])) {
    if (!__builtin_amdgcn_readfirstlane(vote[1])) return;
    atomicMax(&vote[2], __builtin_bit_cast(uint32_t, most));
    atomicMin(&vote[3], __builtin_bit_cast(uint32_t, smallest));
    __syncthreads();
    const float largest_operand = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(vote[2]));
    const float smallest_result = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(vote[3]));
    if (smallest_result >= (float)K * 0x1p-99f * largest_operand) return;
  }
  f32x16 sum[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) sum[i][j][e] = 0.0f;
  const float *arow[MT], *bcol[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int64_t r = 32 * i + (l & 31), last = M - 1 - m0;
    arow[i] = A + (m0 + (r < last ? r : last)) * lda;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int64_t c = n0 + w * 32 * NT + 32 * j + (l & 31);
    bcol[j] = B + (c < N ? c : N - 1);
  }
  // Eight of k at a time, a lane 4 in a row; the next ones are fetched under the multiplies (2048 cycles for 128
  // rows).  The last 1..8 of k element by element.
  struct Eight {
    float a[MT][4], b[NT][4];
  };
  auto fetch = [&](Eight& x, int k) {
#pragma unroll
    for (int i = 0; i < MT; ++i) __builtin_memcpy(x.a[i], arow[i] + k, 16);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) x.b[j][e] = bcol[j][(int64_t)(k + e) * ldb];
  };
  auto multiply = [&](const Eight& x) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.b[j][e], x.a[i][e], sum[i][j], 0, 0, 0);
  };
  const int eights = (K - 1) / 8, k_lane = 4 * (l >> 5);  // (K is 17 at least)
  Eight x, next;
  fetch(x, k_lane);
  for (int g = 0; g < eights; ++g) {
    fetch(next, 8 * (g + 1 < eights ? g + 1 : g) + k_lane);
    __builtin_amdgcn_sched_barrier(0);  // (the loads stay in front of the multiplies)
    multiply(x);
    __builtin_amdgcn_sched_barrier(0);
    x = next;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int k = 8 * eights + k_lane + e, kc = k < K ? k : K - 1;
#pragma unroll
    for (int i = 0; i < MT; ++i) x.a[i][e] = k < K ? arow[i][kc] : 0.0f;
#pragma unroll
    for (int j = 0; j < NT; ++j) x.b[j][e] = k < K ? bcol[j][(int64_t)kc * ldb] : 0.0f;
  }
  multiply(x);
  store_tile<MathF32, MT, 4, S::TILE_M, true, NT>(epi, sum, lds, w, 0, w, m0, n0, M, N, 0.0f, 0.0f);
}

}  // namespace tile
}  // namespace cig
