// GEMM of a batch of rows on tiles of 64 or 128 rows x 64 columns, one round of them, all of k in one workgroup.
//
// What bounds these calls: a compute unit takes 50 to 55 KB/us of operands here (111 where every line is in its L2:
// lines that come from memory hold up those behind them), also with half of the units at work; and, where k is cut
// to fill the chip with 256-column tiles, the partial sums and the launch that adds them up (5 to 8 us).  Tiles
// of 64 columns fill it with whole k: 4 x 64 tiles of 64 rows serve 256 x 4096 where mfma_tile.h has 64 tiles
// and cuts k in four.  Wider outputs or longer k are that kernel's, whose 256 columns share each fetch of A.  us,
// there -> here: bf16 229 x 2752 x 1984 17.4 -> 11.9, 1097 x 1664 x 1664 19.0 -> 13.6, 113 x 14464 x 2624 29.0 ->
// 22.9; int8 with scales 256 x 4096 x 4096 17.3 -> 12.7, 512 x 4096 x 4096 22.8 -> 17.0.
// Tried and not kept: K ranges joined inside (by the tile's last workgroup; a few calls gained), tiles of 256 rows
// (256 x 8192 x 8192 over two ranges 59.7 us, 51.7 on the tile kernel), K x N int8 (whose 64-byte rows are half
// lines: as fast as the tile kernel at best), a ring of 10 for 64 rows (no difference), workgroups that begin at
// different stages (none), waves that move only A or only B through rings of their own (256 x 4096 x 4096 21.7 ->
// 28.2).
//
// Workgroup = 512 lanes = 8 waves, 2 (rows) x 4 (k): a stage is 128 bytes of k (64 halves, 128 int8), of which
// each wave multiplies one k-step of 32 MT rows x 64 columns.  Stages of A [rows][128 B] and B ([64 n][128 B] or
// [64 k][64 n] halves) go to LDS by LDS-DMA into a ring of RING slots, all of them in flight but the one whose
// fragments are in registers; one barrier a stage.  The four sums meet in LDS.
#include "epilogues.h"
#include "kpiece.h"
#include "mfma_tile.h"
#include "panel_plan.h"

namespace cig {
namespace panel {
namespace {

template <int MT>
struct Geo {
  static constexpr int ROWS = 64 * MT;
  static constexpr int A_BYTES = ROWS * PB, SLOT = A_BYTES + TN * PB;
  static constexpr int RING = MT == 2 ? 6 : 8;
  static constexpr int LDS_BYTES = RING * SLOT;
  static constexpr int PER = MT + 1;           // DMA instructions of a wave per stage
  static constexpr int SUM_LD = TN + 4;        // floats per row of the sums in LDS
  static constexpr int SUM_BYTES = ROWS * SUM_LD * 4;
  static_assert(2 * SUM_BYTES <= LDS_BYTES && LDS_BYTES <= 160 * 1024, "");
};

// lda, ldb in bytes.  grid.x = tiles_m * tiles_n.  k_bytes is a multiple of 16: what is missing of the last stage
// is fetched as zeros.
template <typename Math, int BMODE, int MT, typename Epi>
__global__ __launch_bounds__(512, 2) void panel_kernel(int M, int N, int tiles_m, int k_bytes,
                                                       const char* __restrict__ A, int64_t lda,
                                                       const char* __restrict__ B, int64_t ldb, Epi epi) {
  typedef typename Math::acc_t acc_t;
  typedef typename Math::scalar_t scalar_t;
  typedef kwaves::BPiece<BMODE> BT;
  typedef Geo<MT> G;
  constexpr int RING = G::RING, SLOT = G::SLOT, PER = G::PER;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int t = threadIdx.x, l = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = w & 1, kg = w >> 1;

  // Workgroups go to the 8 XCDs round-robin: each gets a contiguous range of logical ids, in which the row
  // tiles of one column tile (they share B's columns) follow each other.
  const int nwg = gridDim.x, xcd = blockIdx.x % 8, local = blockIdx.x / 8;
  const int base = nwg / 8, rem8 = nwg % 8;
  const int id = xcd * base + (xcd < rem8 ? xcd : rem8) + local;
  const int tm = __builtin_amdgcn_readfirstlane(id % tiles_m);
  const int tn = __builtin_amdgcn_readfirstlane(id / tiles_m);
  const int64_t m0 = (int64_t)tm * G::ROWS, n0 = (int64_t)tn * TN;

  const int stages = (k_bytes + PB - 1) / PB;
  const int last_bytes = k_bytes - (stages - 1) * PB;  // of k in the last stage

  const char* const a_tile = kwaves::uniform(A + m0 * lda);
  const char* b_tile;
  int64_t b_step;
  if constexpr (BMODE == tile::B_NK) {
    b_tile = kwaves::uniform(B + n0 * ldb);
    b_step = PB;
  } else {
    b_tile = kwaves::uniform(B + n0 * Math::ELEM_BYTES);
    b_step = (int64_t)(PB / Math::ELEM_BYTES) * ldb;
  }
  // rows past M (N x K: past N) re-read the last valid row, chunks past N the last valid one; what they
  // produce is never stored
  const int a_last = (int)(M - 1 - m0 < G::ROWS - 1 ? M - 1 - m0 : G::ROWS - 1);
  const int n_left = (int)(N - n0 < TN ? N - n0 : TN);
  const int b_last = BMODE == tile::B_NK ? n_left - 1 : (n_left * Math::ELEM_BYTES + 15) / 16 - 1;
  // A instruction w MT + i: rows 8 (w MT + i) ..; B instruction w: 1 KiB of the piece
  uint32_t a_voff[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r = 8 * (w * MT + i) + (l >> 3);
    a_voff[i] =
        (uint32_t)((int64_t)(r < a_last ? r : a_last) * lda + (((l & 7) ^ tile::pair_swz(r)) << 4));
  }
  const uint32_t b_voff = BT::dma_src(w, l, ldb, b_last);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  // (asm, so that the compiler's wait counts do not know the transfers: see mfma_tile.h)
  auto dma16 = [&](const char* from, uint32_t voff, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(dst), "v"(voff), "s"(from)
                 : "m0");
  };
  auto dma16z = [&](const char* from, uint32_t voff, uint32_t dst, bool zero) {
    const char* const src = zero ? reinterpret_cast<const char*>(tile::g_zero_chunk) : from + voff;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(dst), "v"(src) : "m0");
  };
  auto issue = [&](int st, uint32_t slot) {
    const char* const a_src = a_tile + (int64_t)st * PB;
    const char* const b_src = b_tile + (int64_t)st * b_step;
    const uint32_t a_dst = lds_base + slot + w * MT * 1024, b_dst = lds_base + slot + G::A_BYTES + w * 1024;
    if (st == stages - 1 && last_bytes < PB) {
      // the first byte of k of the lane's piece of B
      const int b_k = BMODE == tile::B_NK ? ((l & 7) ^ tile::pair_swz(8 * w + (l >> 3))) << 4
                                          : (8 * w + (l >> 3)) * Math::ELEM_BYTES;
      dma16z(b_src, b_voff, b_dst, b_k >= last_bytes);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int r = 8 * (w * MT + i) + (l >> 3);
        dma16z(a_src, a_voff[i], a_dst + i * 1024, (((l & 7) ^ tile::pair_swz(r)) << 4) >= last_bytes);
      }
    } else {
      dma16(b_src, b_voff, b_dst);
#pragma unroll
      for (int i = 0; i < MT; ++i) dma16(a_src, a_voff[i], a_dst + i * 1024);
    }
  };

  acc_t acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

  struct Frags {
    u32x4 a[MT], b[2];
  };
  Frags f[2];
  const int a_at = tile::pair_off(wm * 32 * MT + (l & 31), 2 * kg + (l >> 5));
  auto read = [&](Frags& x, uint32_t slot) {
    const char* const s = lds + slot;
#pragma unroll
    for (int j = 0; j < 2; ++j) x.b[j] = BT::frag(s + G::A_BYTES, 32 * j, kg, l);
    // (32 rows further the swizzle is the same)
#pragma unroll
    for (int i = 0; i < MT; ++i) x.a[i] = *reinterpret_cast<const u32x4*>(s + a_at + i * 32 * PB);
  };
  // vmcnt(n), everything else unconstrained
  auto wait = [](auto n_) {
    constexpr int n = decltype(n_)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70 | (n & 15) | ((n >> 4) << 14));
  };
  // at most `rem` whole stages still in flight
  auto wait_stages = [&](int rem) {
    if (rem >= RING - 2) return wait(std::integral_constant<int, (RING - 2) * PER>{});
    if (rem >= 3) return wait(std::integral_constant<int, 3 * PER>{});
    if (rem >= 1) return wait(std::integral_constant<int, PER>{});
    wait(std::integral_constant<int, 0>{});
  };
  static_assert((RING - 1) * PER < 64, "vmcnt is a 6-bit counter");

#pragma unroll
  for (int s = 0; s < RING; ++s)
    if (s < stages) issue(s, s * SLOT);
  // (stage 0 landed)
  if (stages >= RING)
    wait(std::integral_constant<int, (RING - 1) * PER>{});
  else
    wait_stages(stages - 1);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  read(f[0], 0);

  uint32_t slot = 0, next = SLOT;
  // Stage s, its fragments in f[CUR]: the next one has landed everywhere; this one's slot is refilled.
  auto stage = [&](int s, auto cur_) {
    constexpr int CUR = decltype(cur_)::value;
    if (s + 1 < stages) {
      wait_stages(stages - 2 - s);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave has read the slot
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (s + RING < stages) issue(s + RING, slot);
      read(f[CUR ^ 1], next);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i][j] = Math::mfma(f[CUR].b[j], f[CUR].a[i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
    slot = next;
    next = next + SLOT == RING * SLOT ? 0 : next + SLOT;
  };
  for (int s = 0; s < stages; s += 2) {
    stage(s, std::integral_constant<int, 0>{});
    if (s + 1 < stages) stage(s + 1, std::integral_constant<int, 1>{});
  }

  // ---- the four sums: (0 + 2) + (1 + 3) --------------------------------------------------------
  // acc[i][j][4 q + e] = C[m0 + 32 (MT wm + i) + l % 32][n0 + 32 j + 8 q + 4 (l / 32) + e]
  typedef __attribute__((ext_vector_type(4))) scalar_t quad_t;
  __syncthreads();  // (every wave has its last fragments; nothing is in flight)
  char* const sums = lds + (kg & 1) * G::SUM_BYTES;
  auto quad_at = [&](int i, int j, int q) {
    return reinterpret_cast<quad_t*>(
        sums + ((wm * 32 * MT + 32 * i + (l & 31)) * G::SUM_LD + 32 * j + 8 * q + 4 * (l >> 5)) * 4);
  };
  auto quad_of = [&](int i, int j, int q) {
    return quad_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
  };
  if (kg >= 2) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) *quad_at(i, j, q) = quad_of(i, j, q);
  }
  __syncthreads();
  if (kg < 2) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) *quad_at(i, j, q) = quad_of(i, j, q) + *quad_at(i, j, q);
  }
  __syncthreads();
  // thread t stores columns 4 (t % 16) .. of rows t / 16 + 32 h
  const int orow = t >> 4, ocol = (t & 15) * 4;
#pragma unroll
  for (int h = 0; h < 2 * MT; ++h) {
    const char* const at = lds + ((orow + 32 * h) * G::SUM_LD + ocol) * 4;
    const quad_t s = *reinterpret_cast<const quad_t*>(at) + *reinterpret_cast<const quad_t*>(at + G::SUM_BYTES);
    const scalar_t sum[4] = {s[0], s[1], s[2], s[3]};
    const int64_t r = m0 + orow + 32 * h, c = n0 + ocol;
    if (r < M && c < N) tile::store_quad_any(epi, r, c, N, sum);
  }
}

template <typename Math, int BMODE, int MT, typename Epi>
void launch_rows(cigemmContext* ctx, int64_t M, int64_t N, int64_t K_bytes, const void* A, int64_t lda_bytes,
                 const void* B, int64_t ldb_bytes, const Epi& epi) {
  typedef Geo<MT> G;
  auto kern = panel_kernel<Math, BMODE, MT, Epi>;
  static std::atomic<uint64_t> lds_set{0};
  if (!ensure_dynamic_lds(ctx, (const void*)kern, G::LDS_BYTES, lds_set)) return;
  const int64_t tiles_m = any::div_up(M, G::ROWS), tiles_n = any::div_up(N, TN);
  ctx->last_tile_rows = G::ROWS;
  ctx->last_k_splits = 1;
  ctx->last_waves = 8;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(512), G::LDS_BYTES, ctx->stream, (int)M, (int)N,
                     (int)tiles_m, (int)K_bytes, static_cast<const char*>(A), lda_bytes,
                     static_cast<const char*>(B), ldb_bytes, epi);
}

template <typename Math, int BMODE, typename Epi>
void launch(cigemmContext* ctx, int rows, int64_t M, int64_t N, int64_t K_bytes, const void* A, int64_t lda_bytes,
            const void* B, int64_t ldb_bytes, const Epi& epi) {
  if (rows == 64)
    launch_rows<Math, BMODE, 1>(ctx, M, N, K_bytes, A, lda_bytes, B, ldb_bytes, epi);
  else
    launch_rows<Math, BMODE, 2>(ctx, M, N, K_bytes, A, lda_bytes, B, ldb_bytes, epi);
}

void set_name(cigemmContext* ctx, const char* dtype, int k_elems, const char* suffix) {
  snprintf(ctx->kernel_name, sizeof(ctx->kernel_name), "%s_mfma_panel_%dx64x%d_w8%s", dtype, ctx->last_tile_rows,
           k_elems, suffix);
  ctx->last_kernel = ctx->kernel_name;
}

// Rows of a tile, 0: another kernel's call.  `ok`: the aligned tile kernel can run it.
int rows_of(const cigemmContext* ctx, bool ok, const Cost& cost, const any::Cost& other, const any::Problem& p) {
  if (!ok || ctx->force_panel_rows < 0 || p.K_bytes > 2147483647LL ||
      any::div_up(p.M, 64) * any::div_up(p.N, TN) > 2147483647LL)
    return 0;
  if (ctx->force_panel_rows > 0) return ctx->force_panel_rows;
  // (a plan of another kernel is imposed)
  if (ctx->force_tile_rows || ctx->force_kwaves) return 0;
  return choose(cost, other, p, ctx->num_cus > 0 ? ctx->num_cus : 256, ctx->workspace ? ctx->ws_partial_bytes : 0);
}

}  // namespace
}  // namespace panel

bool launch_panel_16(cigemmContext* ctx, bool bf16, int64_t M, int64_t N, int64_t K, const uint16_t* A, int64_t lda,
                     const uint16_t* B, int64_t ldb, uint16_t* C, int64_t ldc) {
  const int rows = panel::rows_of(ctx, tile_16_ok(M, N, K, A, lda, B, ldb, C, ldc), panel::COST_16, any::COST_16,
                                  any::Problem{M, N, K * 2, 2, 2, false, false, false});
  if (!rows) return false;
  if (bf16)
    panel::launch<tile::MathBF16, tile::B_KN16>(ctx, rows, M, N, K * 2, A, lda * 2, B, ldb * 2,
                                                EpiStore16x4<BF16>{C, ldc});
  else
    panel::launch<tile::MathF16, tile::B_KN16>(ctx, rows, M, N, K * 2, A, lda * 2, B, ldb * 2,
                                               EpiStore16x4<F16>{C, ldc});
  panel::set_name(ctx, bf16 ? "bf16" : "f16", 64, "");
  return true;
}

// (the accumulator dump is left to the other kernels)
bool launch_panel_i8_nk(cigemmContext* ctx, int64_t M, int64_t N, int64_t K, const int8_t* A, int64_t lda,
                        const int8_t* B, int64_t ldb, int32_t* C, int64_t ldc, const DequantArgs* dq) {
  const int rows = panel::rows_of(
      ctx, tile::i8_tile_ok(M, N, K, A, lda, B, ldb, true, C, ldc, dq) && !(dq && dq->acc_out), panel::COST_I8_NK,
      any::COST_I8_NK, any::Problem{M, N, K, 1, dq && dq->out_bf16 ? 2 : 4, dq != nullptr, false, false});
  if (!rows) return false;
  if (!dq)
    panel::launch<tile::MathI8, tile::B_NK>(ctx, rows, M, N, K, A, lda, B, ldb, EpiStoreI32x4{C, ldc});
  else if (dq->out_bf16)
    panel::launch<tile::MathI8, tile::B_NK>(ctx, rows, M, N, K, A, lda, B, ldb,
                                            EpiDequantX4<true, false>{dq->out, dq->ldo, dq->sa, dq->sb, dq->sa_vec,
                                                                      dq->sb_vec, nullptr, 0});
  else
    panel::launch<tile::MathI8, tile::B_NK>(ctx, rows, M, N, K, A, lda, B, ldb,
                                            EpiDequantX4<false, false>{dq->out, dq->ldo, dq->sa, dq->sb, dq->sa_vec,
                                                                       dq->sb_vec, nullptr, 0});
  panel::set_name(ctx, "i8", 128, dq ? "_nk_dequant" : "_nk");
  return true;
}

}  // namespace cig
