// How the quantized BatchMatMul kernels bring an operand into LDS: 64 x 64 byte tiles, k-contiguous per output row / column.
#ifndef ITEXHIP_QBMM_STAGE_HPP_
#define ITEXHIP_QBMM_STAGE_HPP_

#include "qbmm_reads.hpp"
#include "qgemm_common.hpp"

namespace itexhip {

// The kernel of row bands (qbmm_band.hip).  Takes the call and enqueues it, or returns false where its rule leaves it to the
// tiles; the arguments are checked and adjacent batch dimensions merged.  `large`: the tiles would be those of 128 rows.
bool qbmm_band(const itexhip_bmm_params& p, int64_t batch, int mode_x, int mode_y, bool large, const int8_t* x, const int8_t* y, void* out,
               hipStream_t st);

namespace {

constexpr int kTile = 64;          // output tile edge and k step
constexpr int kLdsStride = 80;     // bytes per LDS row: 64 + 16, keeps the 16-byte fragment reads aligned
constexpr int kBmmThreads = 256;

// How an operand is read, each by itself.  kBytes: rows too short for a load (and an empty K): byte by byte, every read
// guarded.  kAligned: aligned 16-byte (KCONT) / 4-byte (transposed) loads that never straddle a bound.  kAny: the same loads
// at whatever byte address they fall on (the hardware takes unaligned vector loads); a load that would cross the end of its
// row starts at the last place inside it and settle_tile shifts the bytes into place once they have arrived.  P.V over 197
// tokens (384 products of 197 x 197 by 197 x 64 to bfloat16): 36.9 us with byte loads (16 per piece), 11.6 us with these.
enum : int { kBytes = 0, kAligned = 1, kAny = 2 };
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));

// One 64 (rows or columns of the output) x 64 (k) byte tile on its way into LDS, k-contiguous there.  The
// global loads (fetch_tile) and the LDS stores (put_tile) are separate so that the next tile's loads are in
// flight while the current one is multiplied.
//   KCONT: the operand is stored [R, K] (k fastest);  else [K, R] (r fastest) and is transposed in put_tile.
template <bool KCONT, int MODE>
__device__ __forceinline__ void fetch_tile(const int8_t* __restrict__ g, int64_t R, int64_t K, int64_t r0, int64_t k0,
                                           int t, uint32_t (&w)[4]) {
  if constexpr (KCONT) {  // thread: row t / 4, 16 consecutive k
    const int64_t row = r0 + (t >> 2), k = k0 + (t & 3) * 16;
    if constexpr (MODE == kAny) {  // (results of rows past R are not stored)
      const v4i v = *reinterpret_cast<const v4i_any*>(g + read_offset_k_fastest(row, k, R, K));
      w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
      return;
    }
    w[0] = w[1] = w[2] = w[3] = 0;
    if (row >= R) return;
    const int8_t* src = g + row * K + k;
    if constexpr (MODE == kAligned) {
      if (k < K) {
        const v4i v = *reinterpret_cast<const v4i*>(src);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
      }
    } else {
#pragma unroll
      for (int b = 0; b < 16; ++b)
        if (k + b < K) w[b >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(src[b])) << (8 * (b & 3));
    }
  } else {  // thread: 4 (k) x 4 (r) bytes; kb = t / 16 picks the k rows, cb = t % 16 the r columns; w[i] = k row i
    const int kb = t >> 4, cb = t & 15;
    const int64_t r = r0 + cb * 4;
    if constexpr (MODE == kAny) {
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const u32_any*>(g + read_offset_r_fastest(r, k0 + kb * 4 + i, R, K));
      return;
    }
    w[0] = w[1] = w[2] = w[3] = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t k = k0 + kb * 4 + i;
      if (k >= K) continue;
      const int8_t* src = g + k * R + r;
      if constexpr (MODE == kAligned) {
        if (r < R) w[i] = *reinterpret_cast<const uint32_t*>(src);
      } else {
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (r + b < R) w[i] |= static_cast<uint32_t>(static_cast<uint8_t>(src[b])) << (8 * b);
      }
    }
  }
}

// kAny: what fetch_tile brought, with the bytes of a piece that crosses a bound moved into place and everything past K
// cleared.  Only the last k tile and the last columns of the operand have such pieces.
template <bool KCONT>
__device__ __forceinline__ void settle_tile(int64_t R, int64_t K, int64_t r0, int64_t k0, int t, uint32_t (&w)[4]) {
  if constexpr (KCONT) {
    if (k0 + kTile <= K) return;
    const int left = static_cast<int>(K - k0) - (t & 3) * 16;  // bytes of this piece inside the row
    if (left >= 16) return;
    const uint32_t shift = left > 0 ? 16 - left : 0;           // 1 .. 15
    v4i v = shift_down(v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]), static_cast<int>(w[3])}, shift);
    if (left <= 0) v = v4i{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = static_cast<uint32_t>(v[i]);
  } else {
    if (r0 + kTile > R) {
      const int over = static_cast<int>(r0 - (R - 4)) + (t & 15) * 4;  // how far the load was moved back
      const uint32_t bits = over > 0 && over < 4 ? over * 8 : 0;       // past the last column: whatever came (not stored)
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] >>= bits;
    }
    if (k0 + kTile > K) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k0 + (t >> 4) * 4 + i >= K) w[i] = 0;
    }
  }
}

template <bool KCONT>
__device__ __forceinline__ void put_tile(uint8_t* __restrict__ lds, int t, const uint32_t (&w)[4]) {
  if constexpr (KCONT) {
    *reinterpret_cast<v4i*>(lds + (t >> 2) * kLdsStride + (t & 3) * 16) =
        v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]), static_cast<int>(w[3])};
  } else {
    const int kb = t >> 4, cb = t & 15;
    uint32_t v[4];
    transpose_4x4(w, v);
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t*>(lds + (cb * 4 + j) * kLdsStride + kb * 4) = v[j];
  }
}

template <int T>
__device__ __forceinline__ float widen(float v) { return v; }
template <int T>
__device__ __forceinline__ float widen(uint16_t bits) {
  return T == ITEXHIP_BFLOAT16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(bits);
}

}  // namespace
}  // namespace itexhip
#endif  // ITEXHIP_QBMM_STAGE_HPP_
