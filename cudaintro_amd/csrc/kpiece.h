// 128 bytes of k of an operand B in LDS, as gemm_kwaves.hip and gemm_panel.hip fetch and read them.
#pragma once
#include "mfma_tile.h"

namespace cig {
namespace kwaves {

// B piece: DMA instruction q fills 1 KiB; lane l fetches the 16 bytes at dma_src from the tile's
// origin (`last` = last valid row (N x K) or 16-byte chunk of a row (K x N)).  frag: the fragment of the
// 32 columns from n0, k-step kk (0..3).
template <int BMODE>
struct BPiece;

template <>
struct BPiece<tile::B_NK> {
  static __device__ __forceinline__ int off(int r, int c) { return tile::pair_off(r, c); }
  static __device__ __forceinline__ uint32_t dma_src(int q, int l, int64_t ld, int last) {
    const int r = 8 * q + (l >> 3);
    return (uint32_t)((int64_t)(r < last ? r : last) * ld + (((l & 7) ^ tile::pair_swz(r)) << 4));
  }
  static __device__ __forceinline__ u32x4 frag(const char* sb, int n0, int kk, int l) {
    return *reinterpret_cast<const u32x4*>(sb + off(n0 + (l & 31), 2 * kk + (l >> 5)));
  }
};

// [64 k][64 n] halves: two rows of 128 bytes span the banks; of the four rows a transposing read
// touches, k and k + 2 take different halves.
template <>
struct BPiece<tile::B_KN16> {
  static constexpr int CHUNKS = 8;
  static __device__ __forceinline__ int swz(int k) { return ((k >> 1) & 1) << 2; }
  static __device__ __forceinline__ int off(int k, int c) { return k * 128 + ((c ^ swz(k)) << 4); }
  static __device__ __forceinline__ uint32_t dma_src(int q, int l, int64_t ld, int last) {
    const int k = 8 * q + (l >> 3), c = (l & 7) ^ swz(k);
    return (uint32_t)((int64_t)k * ld + ((c < last ? c : last) << 4));
  }
  static __device__ __forceinline__ u32x4 frag(const char* sb, int n0, int kk, int l) {
    const int k = 16 * kk + 8 * (l >> 5) + ((l & 15) >> 2);
    const int n = n0 + 16 * ((l >> 4) & 1) + 4 * (l & 3);
    const int sub = ((n >> 2) & 1) * 8;
    typedef tile::lds_i16x4 p_t;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((p_t*)(sb + off(k, n >> 3) + sub));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((p_t*)(sb + off(k + 4, n >> 3) + sub));
    return __builtin_shufflevector(__builtin_bit_cast(u32x2, lo), __builtin_bit_cast(u32x2, hi), 0, 1,
                                   2, 3);
  }
};

// [128 k][64 n] bytes: four rows of 64 bytes span the banks; of the eight rows a transposing read
// touches, k and k + 4 take different halves.
template <>
struct BPiece<tile::B_KN8> {
  static constexpr int CHUNKS = 4;
  static __device__ __forceinline__ int swz(int k) { return ((k >> 2) & 1) << 1; }
  static __device__ __forceinline__ int off(int k, int c) { return k * 64 + ((c ^ swz(k)) << 4); }
  static __device__ __forceinline__ uint32_t dma_src(int q, int l, int64_t ld, int last) {
    const int k = 16 * q + (l >> 2), c = (l & 3) ^ swz(k);
    return (uint32_t)((int64_t)k * ld + ((c < last ? c : last) << 4));
  }
  static __device__ __forceinline__ u32x4 frag(const char* sb, int n0, int kk, int l) {
    const int k = 32 * kk + 16 * (l >> 5) + ((l & 15) >> 1);
    const int n = n0 + 16 * ((l >> 4) & 1) + 8 * (l & 1);
    const int sub = ((n >> 3) & 1) * 8;
    typedef tile::lds_i32x2 p_t;
    const i32x2 lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((p_t*)(sb + off(k, n >> 4) + sub));
    const i32x2 hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((p_t*)(sb + off(k + 8, n >> 4) + sub));
    return __builtin_shufflevector(__builtin_bit_cast(u32x2, lo), __builtin_bit_cast(u32x2, hi), 0, 1,
                                   2, 3);
  }
};

// [32 k][32 n] floats.  A read takes 32 columns of two rows k and k + 4, each half of the banks: row k
// sits at k ^ (bit 2 of k), so that the two have different parities.
template <>
struct BPiece<tile::B_KN32> {
  static constexpr int CHUNKS = 8;
  static __device__ __forceinline__ int row(int k) { return k ^ ((k >> 2) & 1); }  // (its own inverse)
  static __device__ __forceinline__ int off(int k, int c) { return row(k) * 128 + (c << 4); }
  static __device__ __forceinline__ uint32_t dma_src(int q, int l, int64_t ld, int last) {
    const int k = row(8 * q + (l >> 3)), c = l & 7;
    return (uint32_t)((int64_t)k * ld + ((c < last ? c : last) << 4));
  }
  static __device__ __forceinline__ u32x4 frag(const char* sb, int, int kk, int l) {
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = *reinterpret_cast<const uint32_t*>(sb + row(8 * kk + 4 * (l >> 5) + e) * 128 + (l & 31) * 4);
    return v;
  }
};

// The same address, known to the compiler as uniform (a scalar base of the DMA instructions).
__device__ __forceinline__ const char* uniform(const char* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const char*)((uint64_t)hi << 32 | lo);
}

}  // namespace kwaves
}  // namespace cig
