// GEMM of a small output: 32 x 64 tiles (fp32: 32 x 32), one workgroup each, whose four waves share out k.
//
// What bounds these calls is latency: the launch, one trip to memory, what one compute unit can take
// from its L2 while most of the others have nothing to do (about 100 KB per us), and, where K is cut,
// the meeting of the ranges.  A 64 x 256 tile of mfma_tile.h makes one unit fetch 320 rows of K; here
// it fetches 96, on four to eight times as many units, and the ranges meet inside the kernel.  us a
// call, there -> here: bf16 33 x 250 x 333 7.0 -> 5.3..6.0 (the host's own pace), 52 x 64 x 2048 9.0 ->
// 6.5, 48 x 4096 x 3776 13.6 -> 10.5, 678 x 128 x 6284 13.9 -> 9.5; int8 N x K 365 x 96 x 853 13.6 ->
// 6.0, K x N 1066 x 320 x 3264 13.3 -> 9.8, 107 x 6208 x 2576 15.7 -> 13.0; 3080 random calls that came
// here (M 17..40000, N 8..16384, K 64..16384) 1.45 times as fast (geometric mean of the kernels inside a
// graph), 18 of them more than 3 % slower, the worst 16 %.  fp32 (against the tile kernel and the
// register-loaded small kernel): 95 x 896 x 1344 17.1 -> 7.8, 22 x 19 x 7616 24.2 -> 8.4, 5812 x 8 x 5568
// 149 -> 28.6; of 5072 calls that came here 53 more than 3 % slower, the worst 27 %; the error against 64
// bits 1.71e-7 from 2.01e-7 (geometric mean over 112 products), at most 3.8e-7 from 6.1e-7.
//
// Workgroup = 256 lanes = 4 waves.  Wave w takes the 128-byte pieces w, w + 4, ... of k (64 halves,
// 128 int8, 32 floats), each through its own LDS slots -- no barrier before the waves' sums meet --:
// A [32 rows][128 B] and B one of [64 n][128 B] (N x K), [64 k][128 B] (K x N, 16-bit), [128 k][64 B]
// (int8), [32 k][128 B] (fp32), moved by LDS-DMA with the bank swizzle on the global side.  Up to
// MAX_SLOTS pieces of a wave are in flight (144 or 128 KiB a workgroup); with more workgroups than units one
// piece per wave, so that three workgroups share a unit.  The four sums meet in LDS in wave order.
//
// K ranges: the grid has `splits` workgroups per tile.  Each stores its sums to the workspace with
// agent-scope stores and counts its arrival at the tile; the one that arrives last adds the ranges up
// in range order (the result does not depend on who that is), applies the epilogue and zeroes the
// counter.  The ordering contract is the decode kernels' (gemm_skinny.hip): partial stores acknowledged
// (vmcnt 0) and a workgroup barrier before the relaxed agent-scope count, agent-scope loads after it;
// nobody waits for another workgroup.
//
// Any M, N, K and any alignment: the last 1..128 bytes of k that are not a whole piece, or whose rows
// are not whole 16-byte pieces, go through registers with every bound checked.
#include "any_plan.h"
#include "epilogues.h"
#include "kpiece.h"
#include "kwaves_plan.h"
#include "mfma_tile.h"

namespace cig {
namespace kwaves {
namespace {

// Tiles of 32 NT columns: fp32, whose matrix instructions take 64 cycles, 32, the others 64.
template <int BMODE>
struct Geo {
  static constexpr int NT = BMODE == tile::B_KN32 ? 1 : 2;
  static constexpr int TN = 32 * NT;
  static constexpr int A_BYTES = TM * PB, B_BYTES = TN * PB;
  static constexpr int SLOT_BYTES = A_BYTES + B_BYTES;  // 8 or 12 KiB
  static constexpr int PER = SLOT_BYTES / 1024;         // DMA instructions per piece
  static constexpr int MAX_SLOTS = NT == 1 ? 4 : 3;     // pieces of a wave in flight
  static constexpr int SUM_LD = TN + 4;                 // floats per row of a wave's sums in LDS
  static_assert(TM * SUM_LD * 4 <= SLOT_BYTES, "a wave's sums fit its first slot");
};

// vmcnt(rem * PER): at most `rem` whole pieces still in flight
template <int PER>
__device__ __forceinline__ void wait_pieces(int rem) {
  static_assert(3 * PER < 64, "vmcnt is a 6-bit counter");
  if (rem >= 3)
    __builtin_amdgcn_s_waitcnt(0x0f70 | ((3 * PER) & 15) | (((3 * PER) >> 4) << 14));
  else if (rem == 2)
    __builtin_amdgcn_s_waitcnt(0x0f70 | ((2 * PER) & 15) | (((2 * PER) >> 4) << 14));
  else if (rem == 1)
    __builtin_amdgcn_s_waitcnt(0x0f70 | (PER & 15) | ((PER >> 4) << 14));
  else
    __builtin_amdgcn_s_waitcnt(0x0f70);
}

// lda, ldb in bytes; slots: pieces of a wave in flight (1..MAX_SLOTS).  `tail`: the last 1..128 bytes of k
// go through registers.  grid.x = tiles_m * tiles_n * splits; range r covers the bytes
// [r * range_bytes, (r + 1) * range_bytes) of k, the last one what is left; range_bytes is a whole
// number of pieces whenever there is more than one range.
template <typename Math, int BMODE, typename Epi>
__global__ __launch_bounds__(256, 3) void kwaves_kernel(
    int M, int N, int tiles_m, int tiles_n, int splits, int range_bytes, int k_total, int tail,
    int slots, const char* __restrict__ A, int64_t lda, const char* __restrict__ B, int64_t ldb,
    Epi epi, uint64_t* __restrict__ partials, uint32_t* __restrict__ counters) {
  typedef typename Math::acc_t acc_t;
  typedef typename Math::scalar_t scalar_t;
  typedef BPiece<BMODE> BT;
  typedef Geo<BMODE> G;
  constexpr int NT = G::NT, TN = G::TN, A_BYTES = G::A_BYTES, SLOT_BYTES = G::SLOT_BYTES;
  constexpr int NB = 4 * NT;  // DMA instructions of a B piece
  constexpr int SUM_LD = G::SUM_LD;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  __shared__ int is_last;
  const int t = threadIdx.x, l = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);

  // Workgroups go to the 8 XCDs round-robin: each gets a contiguous range of logical ids, in which
  // the row tiles of one column tile (they share B's panel) follow each other and K ranges are
  // outermost (the tiles of one range share A's columns).
  const int nwg = gridDim.x, xcd = blockIdx.x % 8, local = blockIdx.x / 8;
  const int base = nwg / 8, rem8 = nwg % 8;
  const int id = xcd * base + (xcd < rem8 ? xcd : rem8) + local;
  const int tm = __builtin_amdgcn_readfirstlane(id % tiles_m);
  const int tn = __builtin_amdgcn_readfirstlane(id / tiles_m % tiles_n);
  const int range = __builtin_amdgcn_readfirstlane(id / (tiles_m * tiles_n));
  const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * TN;

  const int k_first = range * range_bytes;
  const int k_here = k_total - k_first < range_bytes ? k_total - k_first : range_bytes;
  const int tail_bytes = tail && range == splits - 1 ? (k_here - 1) % PB + 1 : 0;
  const int pieces = (k_here - tail_bytes) / PB;  // whole ones
  const int mine = pieces > w ? (pieces - w + WAVES - 1) / WAVES : 0;

  const char* const a_tile = uniform(A + m0 * lda + k_first);
  const char* b_tile;
  int64_t b_step;
  if constexpr (BMODE == tile::B_NK) {
    b_tile = uniform(B + n0 * ldb + k_first);
    b_step = PB;
  } else {
    b_tile = uniform(B + (int64_t)(k_first / Math::ELEM_BYTES) * ldb + n0 * Math::ELEM_BYTES);
    b_step = (int64_t)(PB / Math::ELEM_BYTES) * ldb;
  }
  // rows past M (N x K: past N) re-read the last valid row, chunks past N the last valid one; what
  // they produce is never stored
  const int a_last = (int)(M - 1 - m0 < TM - 1 ? M - 1 - m0 : TM - 1);
  const int n_left = (int)(N - n0 < TN ? N - n0 : TN);
  const int b_last = BMODE == tile::B_NK ? n_left - 1 : (n_left * Math::ELEM_BYTES + 15) / 16 - 1;
  uint32_t a_voff[4], b_voff[NB];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 8 * q + (l >> 3);
    a_voff[q] = (uint32_t)((int64_t)(r < a_last ? r : a_last) * lda +
                           (((l & 7) ^ tile::pair_swz(r)) << 4));
  }
#pragma unroll
  for (int q = 0; q < NB; ++q) b_voff[q] = BT::dma_src(q, l, ldb, b_last);
  char* const own = lds + w * slots * SLOT_BYTES;  // this wave's slots
  const uint32_t own_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)own;
  auto dma16 = [&](const char* from, uint32_t voff, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_dst), "v"(voff), "s"(from)
                 : "m0");
  };
  // fetches this wave's i-th piece into `slot`
  auto issue = [&](int i, int slot) {
    const int p = w + WAVES * i;
    const char* const a_src = a_tile + (int64_t)p * PB;
    const char* const b_src = b_tile + (int64_t)p * b_step;
    const uint32_t dst = own_base + slot * SLOT_BYTES;
#pragma unroll
    for (int q = 0; q < NB; ++q) dma16(b_src, b_voff[q], dst + A_BYTES + q * 1024);
#pragma unroll
    for (int q = 0; q < 4; ++q) dma16(a_src, a_voff[q], dst + q * 1024);
  };

  acc_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[j][e] = 0;
  struct Frags {
    u32x4 a[4], b[4][NT];
  };
  auto read = [&](Frags& f, const char* sa) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      f.a[kk] = *reinterpret_cast<const u32x4*>(sa + tile::pair_off(l & 31, 2 * kk + (l >> 5)));
#pragma unroll
      for (int j = 0; j < NT; ++j) f.b[kk][j] = BT::frag(sa + A_BYTES, 32 * j, kk, l);
    }
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if constexpr (Math::SUBSTEPS == 1) {
          acc[j] = Math::mfma(f.b[kk][j], f.a[kk], acc[j]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[j] = Math::mfma(Math::afrag(f.b[kk][j], e), Math::afrag(f.a[kk], e), acc[j]);
        }
      }
  };

#pragma unroll
  for (int i = 0; i < G::MAX_SLOTS; ++i)
    if (i < slots && i < mine) issue(i, i);
  int slot = 0;
  for (int i = 0; i < mine; ++i) {
    const int rem = mine - 1 - i < slots - 1 ? mine - 1 - i : slots - 1;
    wait_pieces<G::PER>(rem);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    Frags f;
    read(f, own + slot * SLOT_BYTES);
    if (i + slots < mine) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
      __builtin_amdgcn_sched_barrier(0);
      issue(i + slots, slot);
    }
    multiply(f);
    slot = slot + 1 == slots ? 0 : slot + 1;
  }

  if (tail_bytes > 0 && w == pieces % WAVES) {
    constexpr int CE = 16 / Math::ELEM_BYTES;
    typedef typename tile::ElemOf<Math::ELEM_BYTES>::type elem_t;
    const elem_t* Ae = reinterpret_cast<const elem_t*>(A + k_first);
    const elem_t* Be = reinterpret_cast<const elem_t*>(
        B + (BMODE == tile::B_NK ? (int64_t)k_first
                                 : (int64_t)(k_first / Math::ELEM_BYTES) * ldb));
    const int64_t lda_e = lda / Math::ELEM_BYTES, ldb_e = ldb / Math::ELEM_BYTES;
    const int64_t k0 = (int64_t)pieces * PB / Math::ELEM_BYTES, k_end = k_here / Math::ELEM_BYTES;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    u32x4 ta[4], tb[NB];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = l + 64 * q;
      ta[q] = tile::load_piece(Ae, lda_e, m0 + (c >> 3), M, k0 + (c & 7) * CE, k_end);
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int c = l + 64 * q;
      if constexpr (BMODE == tile::B_NK)
        tb[q] = tile::load_piece(Be, ldb_e, n0 + (c >> 3), N, k0 + (c & 7) * CE, k_end);
      else
        tb[q] = tile::load_piece(Be, ldb_e, k0 + c / BT::CHUNKS, k_end, n0 + (c % BT::CHUNKS) * CE, N);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = l + 64 * q;
      *reinterpret_cast<u32x4*>(own + tile::pair_off(c >> 3, c & 7)) =
          tile::trim_piece<elem_t>(ta[q], m0 + (c >> 3), M, k0 + (c & 7) * CE, k_end);
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int c = l + 64 * q;
      if constexpr (BMODE == tile::B_NK)
        *reinterpret_cast<u32x4*>(own + A_BYTES + BT::off(c >> 3, c & 7)) =
            tile::trim_piece<elem_t>(tb[q], n0 + (c >> 3), N, k0 + (c & 7) * CE, k_end);
      else
        *reinterpret_cast<u32x4*>(own + A_BYTES + BT::off(c / BT::CHUNKS, c % BT::CHUNKS)) =
            tile::trim_piece<elem_t>(tb[q], k0 + c / BT::CHUNKS, k_end, n0 + (c % BT::CHUNKS) * CE, N);
    }
    // (LDS serves a wave's instructions in order; the reads must not be moved above the writes)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    Frags f;
    read(f, own);
    multiply(f);
  }

  // The waves' sums, each in its wave's first slot, meet in wave order: thread t holds NT quads of
  // columns 4 (t % QPR).., rows t / QPR + h * ROWS.  acc[j][4q + e] = C[l % 32][32 j + 8 q + 4 g + e].
  typedef __attribute__((ext_vector_type(4))) scalar_t quad_t;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's fragments are in registers
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const quad_t v = {acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
      *reinterpret_cast<quad_t*>(own + ((l & 31) * SUM_LD + 32 * j + 8 * q + 4 * (l >> 5)) * 4) = v;
    }
  __syncthreads();
  constexpr int QPR = TN / 4, ROWS = 256 / QPR;
  const int orow = t / QPR, ocol = (t % QPR) * 4;
  scalar_t sum[NT][4];
#pragma unroll
  for (int h = 0; h < NT; ++h) {
    const char* at = lds + ((orow + ROWS * h) * SUM_LD + ocol) * 4;
    quad_t s = *reinterpret_cast<const quad_t*>(at);
#pragma unroll
    for (int ww = 1; ww < WAVES; ++ww)
      s += *reinterpret_cast<const quad_t*>(at + ww * slots * SLOT_BYTES);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[h][e] = s[e];
  }

  if (splits > 1) {
    // word x of thread t at x * 256 + t of the range's 4 NT KiB
    constexpr int NX = 2 * NT, WORDS = NX * 256;
    const int tile_id = tn * tiles_m + tm;
    uint64_t* const tile_part = partials + (int64_t)tile_id * splits * WORDS + t;
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const uint64_t lo = __builtin_bit_cast(uint32_t, sum[x / 2][x % 2 * 2]);
      const uint64_t hi = __builtin_bit_cast(uint32_t, sum[x / 2][x % 2 * 2 + 1]);
      __hip_atomic_store(tile_part + (int64_t)range * WORDS + x * 256, lo | hi << 32,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): every partial store has been acknowledged
    __syncthreads();
    if (t == 0) {
      const uint32_t old = __hip_atomic_fetch_add(counters + tile_id, 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
      is_last = old == (uint32_t)(splits - 1);
    }
    __syncthreads();
    if (!is_last) return;
#pragma unroll
    for (int h = 0; h < NT; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[h][e] = 0;
    // (the loads of eight ranges are issued back to back before the first addition waits)
    for (int r0 = 0; r0 < splits; r0 += 8) {
      uint64_t v[8][NX];
#pragma unroll
      for (int b = 0; b < 8; ++b)
        if (r0 + b < splits) {
#pragma unroll
          for (int x = 0; x < NX; ++x)
            v[b][x] = __hip_atomic_load(tile_part + (int64_t)(r0 + b) * WORDS + x * 256,
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
      for (int b = 0; b < 8; ++b)
        if (r0 + b < splits) {
#pragma unroll
          for (int x = 0; x < NX; ++x) {
            sum[x / 2][x % 2 * 2] += __builtin_bit_cast(scalar_t, (uint32_t)v[b][x]);
            sum[x / 2][x % 2 * 2 + 1] += __builtin_bit_cast(scalar_t, (uint32_t)(v[b][x] >> 32));
          }
        }
    }
    if (t == 0) __hip_atomic_store(counters + tile_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

#pragma unroll
  for (int h = 0; h < NT; ++h) {
    const int64_t r = m0 + orow + ROWS * h, c = n0 + ocol;
    if (r < M && c < N) tile::store_quad_any(epi, r, c, N, sum[h]);
  }
}

// k and the rows of a K x N operand are whole pieces: nothing goes through registers.
bool is_whole(int64_t K_bytes, int64_t n_bytes, bool b_nk) {
  return K_bytes % PB == 0 && (b_nk || n_bytes % 16 == 0);
}

template <typename Math, int BMODE, typename Epi>
void launch(cigemmContext* ctx, Plan plan, int64_t M, int64_t N, int64_t K_bytes, const void* A,
            int64_t lda_bytes, const void* B, int64_t ldb_bytes, const Epi& epi) {
  typedef Geo<BMODE> G;
  auto kern = kwaves_kernel<Math, BMODE, Epi>;
  static std::atomic<uint64_t> lds_set{0};
  if (!ensure_dynamic_lds(ctx, (const void*)kern, WAVES * G::MAX_SLOTS * G::SLOT_BYTES, lds_set)) return;
  const int tiles_m = (int)((M + TM - 1) / TM), tiles_n = (int)((N + G::TN - 1) / G::TN);
  int64_t range_stages = 0;
  const int splits = tile::k_ranges(K_bytes, plan.splits, &range_stages);
  const int64_t range_bytes = splits > 1 ? range_stages * tile::KB : K_bytes;
  const bool whole = is_whole(K_bytes, N * Math::ELEM_BYTES, BMODE == tile::B_NK);
  const int64_t wgs = (int64_t)tiles_m * tiles_n * splits;
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const int slots = wgs <= cus ? G::MAX_SLOTS : 1;
  ctx->last_tile_rows = TM;
  ctx->last_k_splits = splits;
  ctx->last_waves = WAVES;
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(256), WAVES * slots * G::SLOT_BYTES, ctx->stream,
                     (int)M, (int)N, tiles_m, tiles_n, splits, (int)range_bytes, (int)K_bytes,
                     whole ? 0 : 1, slots, static_cast<const char*>(A), lda_bytes,
                     static_cast<const char*>(B), ldb_bytes, epi,
                     static_cast<uint64_t*>(ctx->workspace),
                     reinterpret_cast<uint32_t*>(static_cast<char*>(ctx->workspace) +
                                                 ctx->ws_partial_bytes));
}

void set_name(cigemmContext* ctx, const char* dtype, int k_elems, const char* suffix, bool any) {
  // (k is always split: over the waves, and over as many ranges as cigemmGetLastPlan reports)
  snprintf(ctx->kernel_name, sizeof(ctx->kernel_name), "%s_mfma_%skwaves_32x64x%d_w4%s_splitk", dtype,
           any ? "any_" : "", k_elems, suffix);
  ctx->last_kernel = ctx->kernel_name;
}

// `ok`: the kernel can run the call; `aligned`: the tile kernel's aligned form can.
Plan plan_of(cigemmContext* ctx, bool ok, const Cost& cost, const any::Cost& other,
             const any::Problem& p, bool aligned, bool b_nk, bool rest) {
  const size_t room = ctx->workspace ? ctx->ws_partial_bytes : 0;
  if (!ok || ctx->force_kwaves < 0 || !fits(p.M, p.N, Plan{1}, room, ctx->ws_counter_bytes))
    return Plan{0};
  if (ctx->force_kwaves > 0) {
    const Plan imposed{ctx->force_kwaves};
    return fits(p.M, p.N, imposed, room, ctx->ws_counter_bytes) ? imposed : Plan{1};
  }
  // (a plan of another kernel is imposed)
  if (ctx->force_tile_rows || ctx->force_panel_rows > 0) return Plan{0};
  if (rest) {
    double est = 0;
    return best(cost, p, false, ctx->num_cus > 0 ? ctx->num_cus : 256, room, ctx->ws_counter_bytes, &est);
  }
  return choose(cost, other, p, is_whole(p.K_bytes, p.N * p.elem, b_nk), aligned,
                ctx->num_cus > 0 ? ctx->num_cus : 256, room, ctx->ws_counter_bytes);
}

void launch_f32(cigemmContext* ctx, Plan plan, int64_t M, int64_t N, int64_t K, const float* A,
                int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc, const BiasAct* ba) {
  if (ba)
    launch<tile::MathF32, tile::B_KN32>(ctx, plan, M, N, K * 4, A, lda * 4, B, ldb * 4,
                                        EpiBiasActAnyF32x4{C, ldc, ba->bias, ba->relu});
  else
    launch<tile::MathF32, tile::B_KN32>(ctx, plan, M, N, K * 4, A, lda * 4, B, ldb * 4,
                                        EpiStoreF32x4{C, ldc});
}

template <int BMODE>
void launch_i8_layout(cigemmContext* ctx, Plan plan, int64_t M, int64_t N, int64_t K, const int8_t* A,
                      int64_t lda, const int8_t* B, int64_t ldb, int32_t* C, int64_t ldc,
                      const DequantArgs* dq) {
  if (!dq)
    launch<tile::MathI8, BMODE>(ctx, plan, M, N, K, A, lda, B, ldb, EpiStoreI32x4{C, ldc});
  else if (dq->out_bf16)
    launch<tile::MathI8, BMODE>(ctx, plan, M, N, K, A, lda, B, ldb,
                                EpiDequantX4<true, false>{dq->out, dq->ldo, dq->sa, dq->sb, dq->sa_vec,
                                                          dq->sb_vec, nullptr, 0});
  else
    launch<tile::MathI8, BMODE>(ctx, plan, M, N, K, A, lda, B, ldb,
                                EpiDequantX4<false, false>{dq->out, dq->ldo, dq->sa, dq->sb,
                                                           dq->sa_vec, dq->sb_vec, nullptr, 0});
}

}  // namespace
}  // namespace kwaves

bool launch_kwaves_16(cigemmContext* ctx, bool bf16, int64_t M, int64_t N, int64_t K,
                      const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, uint16_t* C,
                      int64_t ldc, bool rest) {
  const bool aligned = tile_16_ok(M, N, K, A, lda, B, ldb, C, ldc);
  const any::Problem call{M, N, K * 2, 2, 2, false, any::rows_apart(A, lda * 2),
                          any::rows_apart(B, ldb * 2)};
  const kwaves::Plan p = kwaves::plan_of(ctx, any::tile_ok(M, rest ? 64 : N, K, 2, lda, ldb, true),
                                         kwaves::COST_16, any::COST_16, call, aligned, false, rest);
  if (!p.splits) return false;
  if (bf16)
    kwaves::launch<tile::MathBF16, tile::B_KN16>(ctx, p, M, N, K * 2, A, lda * 2, B, ldb * 2,
                                                 EpiStore16x4<BF16>{C, ldc});
  else
    kwaves::launch<tile::MathF16, tile::B_KN16>(ctx, p, M, N, K * 2, A, lda * 2, B, ldb * 2,
                                                EpiStore16x4<F16>{C, ldc});
  kwaves::set_name(ctx, bf16 ? "bf16" : "f16", 64, "", !aligned);
  return true;
}

bool launch_kwaves_f32(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const float* A,
                       int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                       const BiasAct* ba, bool rest) {
  const size_t room = ctx->workspace ? ctx->ws_partial_bytes : 0;
  kwaves::Plan p{1};
  if (!any::tile_ok(M, rest ? 64 : N, K, 4, lda, ldb, true) || ctx->force_kwaves < 0 ||
      !kwaves::fits(M, N, p, room, ctx->ws_counter_bytes, kwaves::TN_F32))
    return false;
  if (ctx->force_kwaves > 0) {
    if (kwaves::fits(M, N, kwaves::Plan{ctx->force_kwaves}, room, ctx->ws_counter_bytes, kwaves::TN_F32))
      p.splits = ctx->force_kwaves;
  } else {
    // (a plan of another kernel is imposed; up to 16 columns and K = 512 the small kernel's 16-column
    // form streams as fast: 20000 x 10 x 512 11.5 against 11.7 us, 2145 x 15 x 320 5.5 against 6.1)
    if (ctx->force_tile_rows || (!rest && K <= 512 && f32_small_is_narrow(M, N, K, A, lda))) return false;
    double est = 0;
    p = kwaves::best_f32(M, N, K, ctx->num_cus > 0 ? ctx->num_cus : 256, room, ctx->ws_counter_bytes,
                         &est);
    if (!p.splits || (!rest && est >= f32_other(ctx, M, N, K, A, lda, B, ldb, C, ldc, ba).us)) return false;
  }
  kwaves::launch_f32(ctx, p, M, N, K, A, lda, B, ldb, C, ldc, ba);
  snprintf(ctx->kernel_name, sizeof(ctx->kernel_name), "f32_mfma_%ssmall_kwaves_32x32x32_w4%s_splitk",
           f32_small_shape_ok(M, N, K, A, lda) ? "" : "any_", ba ? "_bias_act" : "");
  ctx->last_kernel = ctx->kernel_name;
  return true;
}

// (the accumulator dump is left to the other kernels)
bool launch_kwaves_i8(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const int8_t* A,
                      int64_t lda, const int8_t* B, int64_t ldb, bool b_nk, int32_t* C, int64_t ldc,
                      const DequantArgs* dq, bool rest) {
  const bool aligned = tile::i8_tile_ok(M, N, K, A, lda, B, ldb, b_nk, C, ldc, dq);
  const any::Problem call{M, N, K, 1, dq && dq->out_bf16 ? 2 : 4, dq != nullptr,
                          any::rows_apart(A, lda), any::rows_apart(B, ldb)};
  const kwaves::Plan p = kwaves::plan_of(
      ctx, any::tile_ok(M, rest ? 64 : N, K, 1, lda, ldb, !b_nk) && !(dq && dq->acc_out),
      b_nk ? kwaves::COST_I8_NK : kwaves::COST_I8_KN, b_nk ? any::COST_I8_NK : any::COST_I8_KN, call,
      aligned, b_nk, rest);
  if (!p.splits) return false;
  if (b_nk)
    kwaves::launch_i8_layout<tile::B_NK>(ctx, p, M, N, K, A, lda, B, ldb, C, ldc, dq);
  else
    kwaves::launch_i8_layout<tile::B_KN8>(ctx, p, M, N, K, A, lda, B, ldb, C, ldc, dq);
  kwaves::set_name(ctx, "i8", 128,
                   dq ? (b_nk ? "_nk_dequant" : "_kn_dequant") : (b_nk ? "_nk" : "_kn"),
                   !aligned);
  return true;
}

int64_t kwaves_rest_columns(const cigemmContext* ctx, int64_t M, int64_t N, int64_t K_bytes, bool f32) {
  // A rest of up to 64 columns costs the tile kernel a column of 256-column tiles, a quarter of them
  // or less used; here 32-row tiles of 32 or 64 columns.  fp32 4095 x 4097 x 4099, one column: 63 us of
  // 64-row tiles over four K ranges and 5 of reduction (977 us the call, 930 here); bf16 4096 x 4104 x 4096
  // 124 -> 115, int8 2048 x 8200 x 1024 36.7 -> 32.1; 17 such sizes 1.06 times as fast, none slower.
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  if (ctx->force_tile_rows || ctx->force_kwaves || K_bytes <= 3 * kwaves::PB ||
      any::div_up(M, tile::BM) * any::div_up(N, tile::BN) <= cus)
    return 0;
  int rows = 0;
  const tile::RoundsPlan r = f32 ? tile::plan_rounds32(M, N, K_bytes, cus, &rows)
                                 : tile::plan_rounds(M, N, cus, tile::TILE_UNITS);
  const int64_t rest = N - r.first_cols;
  if (!r.first_cols || rest > 64) return 0;
  const int64_t tiles = any::div_up(M, kwaves::TM) * any::div_up(rest, f32 ? kwaves::TN_F32 : kwaves::TN);
  return tiles <= 3 * (int64_t)cus ? r.first_cols : 0;
}

void name_rest_columns(cigemmContext* ctx, const char* first) {
  char name[sizeof(ctx->kernel_name)];
  snprintf(name, sizeof(name), "%s+%dx%d", first, kwaves::TM,
           strncmp(first, "f32", 3) ? kwaves::TN : kwaves::TN_F32);
  memcpy(ctx->kernel_name, name, sizeof(name));
  ctx->last_kernel = ctx->kernel_name;
}

}  // namespace cig
